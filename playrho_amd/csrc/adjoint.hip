// Hand-written adjoint of the regular step's contact solve and integration
// (SolveRegIslandViaGS, AabbTreeWorld.cpp:1563-1682) for worlds of disks
// against each other and against static edges/polygons: one-point manifolds
// of type circles or face A.  The active set of each step is held fixed as
// recorded by the forward pass (k_step_worlds_tape): which contacts touch and
// form which islands, the clamp branches of every Gauss-Seidel update, the
// iteration counts of the early exits.  Within it every differentiable
// dependence is followed:
//
//   velocity integration        v' = (v + h a) / (1 + h damping)   (Body.cpp:290-309)
//   constraint creation         normal, points, effective masses and the
//                               restitution bias from positions and v'
//                               (WorldManifold.cpp:37-130, VelocityConstraint.cpp:81-185)
//   warm start                  (AabbTreeWorld.cpp:230-274)
//   Gauss-Seidel updates        tangent (friction clamp) then normal
//                               (ContactSolver.cpp:337-454)
//   position integration        (AabbTreeWorld.cpp:176-188)
//   position solver             (ContactSolver.cpp:494-643, PositionSolverManifold.cpp:42-121)
//   impulse carry-over          manifold impulses warm-start the next step
//   material mixing             friction sqrt(fA fB), restitution max(eA, eB) (Contact.hpp:57-69)
//
// One launch reverses one recorded step for every world: one wavefront per
// world, one lane per update of a round (updates that share no moving body).
#include "adjoint_dual.hpp"
#include "layout.hpp"
#include "step_device.hpp"

namespace prxd {

using prx::AdjState;
using prx::Tape;

__device__ __forceinline__ V2 v2(float4 a) { return V2{a.x, a.y}; }
__device__ __forceinline__ V2 perp_grad(V2 c) { return V2{c.y, -c.x}; }  // d dot(revperp(r), c) / dr

__device__ __forceinline__ void add_body(float4* p, V2 v, float w) {
    float4 a = *p;
    a.x += v.x;
    a.y += v.y;
    a.z += w;
    *p = a;
}

// ---------------------------------------------------------------------------
// Reverse rounds.  A step's solver updates are reversed in the opposite of
// their recorded order, but only updates that share a moving body depend on
// one another.  An update's level is one more than the last level that touched
// either of its bodies (bodies with zero inverse mass and inertia order
// nothing); the updates of a level touch distinct moving bodies, so they are
// reversed together, levels from the last to the first, and every sum is
// formed in the order the serial walk forms it.  The plan covers all of a
// world's islands at once; an update takes part in the iterations its island
// ran.

// Levels of items 0..n-1 in recorded order (bodies(k): the moving bodies of
// item k, -1 for none), then rounds of at most `width` items of one level:
// round r is order[start[r]..start[r + 1]).  last: a table of nb ints; lvl: n
// ints of scratch.  Run by one wavefront.  period: the most rounds that any
// body's items span; iterations started that many rounds apart still reach
// every body in order, so they can be reversed side by side.
struct RoundPlan {
    int rounds, period;
};
template <class F>
__device__ __forceinline__ RoundPlan plan_rounds(int n, int nb, int width, int lane, F bodies, int* last, int* lvl, int* order,
                                           int* start) {
    auto fence = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup"); };
    for (int b = lane; b < nb; b += kWave) last[b] = 0;
    fence();
    int levels = 0;
    for (int base = 0; base < n; base += kWave) {
        int2 ab{-1, -1};
        if (base + lane < n) ab = bodies(base + lane);
        const int cnt = (n - base < kWave) ? n - base : kWave;
        int mine = 0;
        for (int j = 0; j < cnt; ++j) {
            const int aj = __builtin_amdgcn_readlane(ab.x, j), bj = __builtin_amdgcn_readlane(ab.y, j);
            const int la = (aj >= 0) ? last[aj] : 0, lb = (bj >= 0) ? last[bj] : 0;
            const int l = ((la > lb) ? la : lb) + 1;
            if (lane == 0) {
                if (aj >= 0) last[aj] = l;
                if (bj >= 0) last[bj] = l;
            }
            fence();
            if (lane == j) mine = l - 1;
            levels = (l > levels) ? l : levels;
        }
        if (base + lane < n) lvl[base + lane] = mine;
    }
    fence();
    // Items by level, then by recorded order: one level after another.  The
    // round of an item replaces its level.
    int rounds = 0, at = 0;
    if (lane == 0) start[0] = 0;
    for (int l = 0; l < levels; ++l) {
        const int first = at;
        for (int base = 0; base < n; base += kWave) {
            const bool in = base + lane < n && lvl[base + lane] == l;
            const unsigned long long m = __ballot(in);
            if (in) {
                const int pos = at + __popcll(m & lanes_below(lane));
                order[pos] = base + lane;
                lvl[base + lane] = -1 - (rounds + (pos - first) / width);
            }
            at += __popcll(m);
        }
        for (int k = first; k < at; k += width) {
            ++rounds;
            if (lane == 0) start[rounds] = (k + width < at) ? k + width : at;
        }
    }
    fence();
    for (int b = lane; b < nb; b += kWave) last[b] = rounds;
    fence();
    for (int k = lane; k < n; k += kWave) {
        const int2 ab = bodies(k);
        if (ab.x >= 0) atomicMin(&last[ab.x], -1 - lvl[k]);
        if (ab.y >= 0) atomicMin(&last[ab.y], -1 - lvl[k]);
    }
    fence();
    int period = 1;
    for (int k = lane; k < n; k += kWave) {
        const int2 ab = bodies(k);
        const int r = -1 - lvl[k];
        if (ab.x >= 0) period = max(period, r - last[ab.x] + 1);
        if (ab.y >= 0) period = max(period, r - last[ab.y] + 1);
    }
    for (int o = 32; o > 0; o >>= 1) period = max(period, __shfl_xor(period, o));
    fence();
    return RoundPlan{rounds, __builtin_amdgcn_readfirstlane(period)};
}

// Iterations of the slots' islands, velocity | position << 16.
__device__ __forceinline__ void slot_iterations(const int4* isl, int nisl, int tid, int threads, int* iters) {
    for (int is = tid; is < nisl; is += threads) {
        const int4 rng = isl[is];
        for (int e = rng.x; e < rng.y; ++e) iters[e] = rng.z | (rng.w << 16);
    }
}
__device__ __forceinline__ int max_iterations(const int4* isl, int nisl, int lane, bool position) {
    int m = 0;
    for (int is = lane; is < nisl; is += kWave) m = max(m, position ? isl[is].w : isl[is].z);
    for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o));
    return __builtin_amdgcn_readfirstlane(m);
}

// Ints of plan scratch per contact slot or joint of a world (AdjState::plan).
static_assert(prx::kAdjPlanInts >= 8, "two plans of levels, order and starts, and the iterations");

// Adds a wavefront's counts to the run's counters: one atomic for each, not
// one for each update (half a million additions to one address a launch took
// most of its time).
__device__ __forceinline__ void add_diag(float* diag, int k, int v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & (kWave - 1)) == 0 && v) atomicAdd(diag + k, float(v));
}

// One wavefront per world, one lane per update of a round.  kLds: the body
// adjoints and the round plan in LDS (36 bytes a body and 12 a contact slot),
// else in global memory.  A round's tape records are read while the round
// before is reversed.  Bound by the latency of one round after another.  1024
// billiards worlds of 64 disks: 0.85 -> 0.21 ms a step against one lane per
// island, the adjoints in global memory and an atomic for each update counted.
template <bool kLds>
__global__ __launch_bounds__(64) void k_adjoint_step(DeviceState d, Tape t, AdjState a, StepParams c) {
    const int w = int(blockIdx.x);
    const int lane = int(threadIdx.x);
    const WorldHeader H = d.hdr[w];
    const int bo = H.body_off, co = H.contact_off, nb = H.nbodies, cap = H.contact_cap;
    const int nisl = t.nisl[w];
    const int4* isl = t.isl + bo + w;
    const int n = nisl > 0 ? isl[nisl - 1].y : 0;
    float4* const X = kLds ? g_smem : a.xbar + bo;
    float4* const V = kLds ? g_smem + nb : a.vbar + bo;
    int* const plan = a.plan + std::size_t(co + H.joint_off) * prx::kAdjPlanInts;
    int* const last = kLds ? reinterpret_cast<int*>(g_smem + 2 * nb) : d.s_stack + 2 * bo;
    int* const order = kLds ? reinterpret_cast<int*>(g_smem + 2 * nb) + nb : plan;
    int* const start = kLds ? order + cap : plan + cap;
    int* const iters = kLds ? start + cap + 1 : plan + 2 * cap + 1;
    int* const lvl = plan + 4 * cap;
    auto vcrec = [&](int e) { return t.vc + (std::size_t(co) + std::size_t(e)) * prx::kTapeVc; };
    // A kinematic disk has no mass but moves at its own velocity, which the
    // contacts it is body B of read: it collects their terms (its mark is the
    // fourth component of its adjoints) and orders the updates that add to them.
    auto kinematic = [&](int b) {
        return (d.bflags[bo + b] & (prx::kSpeedable | prx::kAccelerable)) == prx::kSpeedable;
    };
    for (int b = lane; b < nb; b += kWave) {
        const float4 xb = a.xbar[bo + b], vb = a.vbar[bo + b];
        const float mark = kinematic(b) ? 1.0f : 0.0f;
        X[b] = float4{xb.x, xb.y, xb.z, mark};
        V[b] = float4{vb.x, vb.y, vb.z, mark};
    }
    // Impulse adjoints carried in from the next step, by contact id: the
    // step's final impulses warm-started the next step where the manifold
    // update after the solve carried them (by ContactFeature, else from the
    // nearest point; the tape's carry map says which).  The next step wrote
    // nothing for contacts it did not solve or that started afresh.
    int unmodelled = 0;
    for (int e = lane; e < n; e += kWave) {
        const float4* vc = vcrec(e);
        const std::uint32_t id = __float_as_uint(vc[10].y);
        const float4 lb = a.lambar[co + int(id)];
        const std::uint32_t cm = t.cmap[co + int(id)];
        const bool carried = ((cm >> 8) & 0xfu) >= 1u && (cm & 0xfu) == 0u;
        a.lamtmp[co + e] = carried ? float2{lb.x, lb.y} : float2{0.0f, 0.0f};
        float4* cb = a.cbar + (std::size_t(co) + e) * 3;
        cb[0] = float4{0, 0, 0, 0};
        cb[1] = float4{0, 0, 0, 0};
        cb[2] = float4{0, 0, 0, 0};
    }
    __syncthreads();
    for (int i = lane; i < cap; i += kWave) a.lambar[co + i] = float4{0.0f, 0.0f, 0.0f, 0.0f};
    slot_iterations(isl, nisl, lane, kWave, iters);
    const RoundPlan rp = plan_rounds(n, nb, kWave, lane, [&](int e) {
        const float4* vc = vcrec(e);
        const float4 ms = vc[8];
        const int bB = __float_as_int(vc[5].z);
        return int2{(ms.x != 0.0f || ms.y != 0.0f) ? __float_as_int(vc[2].w) : -1,
                    (ms.z != 0.0f || ms.w != 0.0f || kinematic(bB)) ? bB : -1};
    }, last, lvl, order, start);
    const int rounds = rp.rounds;
    __syncthreads();
    // Slot of the lane in round r of iteration `it` (-1: past the first pass),
    // -1 for none.
    auto slot_at = [&](int it, int r, bool position) {
        if (it < 0) return -1;
        const int pos = start[r] + lane;
        if (pos >= start[r + 1]) return -1;
        const int e = order[pos];
        return it < (position ? iters[e] >> 16 : iters[e] & 0xffff) ? e : -1;
    };

    // Position solver, reversed.
    int posUpdates = 0;
    {
        struct Rec {
            float4 v0, v2, v5, v8, v9, v10, g0, g1;
        };
        auto fetch = [&](int e, int it, Rec& r) {
            if (e < 0) return;
            const float4* vc = vcrec(e);
            const float4* g = t.ngs + ((std::size_t(co) + e) * std::size_t(t.itP) + it) * 2;
            r = Rec{vc[0], vc[2], vc[5], vc[8], vc[9], vc[10], g[0], g[1]};
        };
        int it = rounds > 0 ? max_iterations(isl, nisl, lane, true) - 1 : -1, r = rounds - 1;
        Rec cur{}, next{};
        int e = slot_at(it, r, true);
        fetch(e, it, cur);
        while (it >= 0) {
            // The round before: the last one of the iteration before.
            if (--r < 0) {
                r = rounds - 1;
                --it;
            }
            const int en = slot_at(it, r, true);
            fetch(en, it, next);
            if (e >= 0) {
                const std::uint32_t type = __float_as_uint(cur.v10.z) & 0xffu;
                const std::uint32_t npts = __float_as_uint(cur.v10.z) >> 8;
                const int bA = __float_as_int(cur.v2.w), bB = __float_as_int(cur.v5.z);
                const float4 ms = cur.v8;
                // Circle centres: a dynamic disk's is its position (disks at
                // the body origin); a static body's point does not move.
                const bool dynA = ms.x != 0.0f || ms.y != 0.0f;
                const V2 pA = dynA ? v2(cur.g0) : V2{cur.v9.x, cur.v9.y};
                const V2 pB = v2(cur.g1);
                const float K = ms.x + ms.z;
                if (npts != 1u || (type != 1u && type != 2u)) unmodelled = 1;
                else ++posUpdates;
                if (npts == 1u && (type == 1u || type == 2u) && K > 0.0f) {
                    const float4 xb4 = X[bB];
                    const bool movB = ms.z != 0.0f || ms.w != 0.0f || xb4.w != 0.0f;
                    const V2 xbA = dynA ? v2(X[bA]) : V2{0.0f, 0.0f}, xbB = v2(xb4);
                    const float s = cur.g0.w;  // separation the forward update used
                    const float inner = c.regResolutionRate * (s + c.linearSlop);
                    const float Cc = -clamp_std(inner, -c.maxLinearCorrection, 0.0f);
                    const bool active = !(inner < -c.maxLinearCorrection) && !(0.0f < inner);
                    const V2 gP = mul(ms.z, xbB) - mul(ms.x, xbA);
                    if (type == 1u) {
                        const V2 dd = pB - pA;
                        const float L = __builtin_sqrtf(magsq(dd));
                        if (L > 0.0f) {
                            const V2 nn2{dd.x / L, dd.y / L};
                            const float Cbar = dot(gP, nn2) / K;
                            const V2 nbar = mul(gP, Cc / K);
                            const float sbar = active ? -c.regResolutionRate * Cbar : 0.0f;
                            const float nn = dot(nn2, nbar);
                            const V2 dbar = mul(nbar - mul(nn2, nn), 1.0f / L) + mul(nn2, sbar);
                            if (dynA) add_body(X + bA, -dbar, 0.0f);
                            if (movB) add_body(X + bB, dbar, 0.0f);
                        }
                    } else {
                        // Face A: A is the polygon (static: its plane and normal
                        // are fixed), B the disk whose centre is the clip point.
                        const V2 nrm = v2(cur.v0);
                        const float Cbar = dot(gP, nrm) / K;
                        const float sbar = active ? -c.regResolutionRate * Cbar : 0.0f;
                        if (movB) add_body(X + bB, mul(nrm, sbar), 0.0f);
                    }
                }
            }
            __syncthreads();
            cur = next;
            e = en;
        }
    }
    // Position integration, reversed: x1 = x0 + h v.
    for (int b = lane; b < nb; b += kWave) {
        if (!t.inisl[bo + b]) continue;
        const float4 xb = X[b];
        add_body(V + b, V2{c.dt * xb.x, c.dt * xb.y}, c.dt * xb.z);
    }
    __syncthreads();
    // Gauss-Seidel sweeps, reversed.
    int velUpdates = 0;
    {
        struct Rec {
            float4 v0, v2, v3, v4, v5, v8, v10, g0, g1;
        };
        auto fetch = [&](int e, int it, Rec& r) {
            if (e < 0) return;
            const float4* vc = vcrec(e);
            const float4* g = t.gs + ((std::size_t(co) + e) * std::size_t(t.itV) + it) * 3;
            r = Rec{vc[0], vc[2], vc[3], vc[4], vc[5], vc[8], vc[10], g[0], g[1]};
        };
        int it = rounds > 0 ? max_iterations(isl, nisl, lane, false) - 1 : -1, r = rounds - 1;
        Rec cur{}, next{};
        int e = slot_at(it, r, false);
        fetch(e, it, cur);
        while (it >= 0) {
            // The round before: the last one of the iteration before.
            if (--r < 0) {
                r = rounds - 1;
                --it;
            }
            const int en = slot_at(it, r, false);
            fetch(en, it, next);
            if (e >= 0 && (__float_as_uint(cur.v10.z) >> 8) == 1u) {
                ++velUpdates;
                const std::size_t slot = std::size_t(co) + e;
                // Sums over the iterations (read late, off the chain through the bodies).
                const float2 lb0 = a.lamtmp[slot];  // (normal, tangent)
                const float4 c0 = a.cbar[slot * 3 + 0], c1 = a.cbar[slot * 3 + 1], c2 = a.cbar[slot * 3 + 2];
                const V2 nrm = v2(cur.v0);
                const V2 tg = fwdperp(nrm);
                const float f = cur.v0.z, ts = cur.v0.w;
                const V2 rA{cur.v3.x, cur.v3.y}, rB{cur.v3.z, cur.v3.w};
                const float nm = cur.v4.z, tm = cur.v4.w, bias = cur.v5.x;
                const float mA = cur.v8.x, iA = cur.v8.y, mB = cur.v8.z, iB = cur.v8.w;
                const int bA = __float_as_int(cur.v2.w), bB = __float_as_int(cur.v5.z);
                const bool movA = mA != 0.0f || iA != 0.0f;
                const V2 vA{cur.g0.x, cur.g0.y}, vB{cur.g1.x, cur.g1.y};
                const float wA = cur.g0.z, wB = cur.g1.z, ltOld = cur.g0.w, lnOld = cur.g1.w;
                // Forward recomputation of this update.
                const V2 cl0 = (vB + mul(revperp(rB), wB)) - (vA + mul(revperp(rA), wA));
                const float vt = dot(cl0, tg);
                const float maxI = f * lnOld;
                const float rawT = ltOld + tm * (ts - vt);
                const bool lowT = rawT < -maxI, highT = !lowT && (maxI < rawT);
                const float ltNew = lowT ? -maxI : (highT ? maxI : rawT);
                const float incT = ltNew - ltOld;
                const V2 PT = mul(incT, tg);
                const V2 vA1 = vA - mul(mA, PT), vB1 = vB + mul(mB, PT);
                const float wA1 = wA - iA * cross(rA, PT), wB1 = wB + iB * cross(rB, PT);
                const V2 cl1 = (vB1 + mul(revperp(rB), wB1)) - (vA1 + mul(revperp(rA), wA1));
                const float vn = dot(cl1, nrm);
                const float rawN = lnOld + nm * (bias - vn);
                const float lnNew = (rawN < 0.0f) ? 0.0f : rawN;
                const float incN = lnNew - lnOld;
                // Adjoints of the outputs (a body that does not move has none
                // that reaches another).
                const float4 zero{0.0f, 0.0f, 0.0f, 0.0f};
                const float4 va4 = movA ? V[bA] : zero, vb4 = V[bB];
                const bool movB = mB != 0.0f || iB != 0.0f || vb4.w != 0.0f;
                V2 vbA = v2(va4), vbB = v2(vb4);
                float wbA = va4.z, wbB = vb4.z;
                float2 lb = lb0;
                V2 nbar{c0.x, c0.y}, rAbar{c0.z, c0.w}, rBbar{c1.x, c1.y}, tbar{c1.z, c1.w};
                float nmbar = c2.x, tmbar = c2.y, biasbar = c2.z, fbar = c2.w;
                // Normal update.
                {
                    const V2 gv = mul(mB, vbB) - mul(mA, vbA);
                    const float ginc = dot(gv, nrm) - iA * wbA * cross(rA, nrm) + iB * wbB * cross(rB, nrm);
                    nbar = nbar + mul(gv, incN) + mul(revperp(rA), -iA * wbA * incN) + mul(revperp(rB), iB * wbB * incN);
                    rAbar = rAbar + mul(perp_grad(nrm), -iA * wbA * incN);
                    rBbar = rBbar + mul(perp_grad(nrm), iB * wbB * incN);
                    const float lnTot = lb.x + ginc;
                    float lnOldBar = -ginc;
                    const float rawBar = (rawN < 0.0f) ? 0.0f : lnTot;
                    lnOldBar += rawBar;
                    nmbar += rawBar * (bias - vn);
                    biasbar += rawBar * nm;
                    const float vnbar = -rawBar * nm;
                    const V2 cbv = mul(nrm, vnbar);
                    nbar = nbar + mul(cl1, vnbar);
                    vbB = vbB + cbv;
                    wbB += cross(rB, cbv);
                    rBbar = rBbar + mul(perp_grad(cbv), wB1);
                    vbA = vbA - cbv;
                    wbA -= cross(rA, cbv);
                    rAbar = rAbar - mul(perp_grad(cbv), wA1);
                    lb.x = lnOldBar;
                }
                // Tangent update.
                {
                    const V2 gv = mul(mB, vbB) - mul(mA, vbA);
                    const float ginc = dot(gv, tg) - iA * wbA * cross(rA, tg) + iB * wbB * cross(rB, tg);
                    tbar = tbar + mul(gv, incT) + mul(revperp(rA), -iA * wbA * incT) + mul(revperp(rB), iB * wbB * incT);
                    rAbar = rAbar + mul(perp_grad(tg), -iA * wbA * incT);
                    rBbar = rBbar + mul(perp_grad(tg), iB * wbB * incT);
                    const float ltTot = lb.y + ginc;
                    float ltOldBar = -ginc;
                    float rawBar = 0.0f, maxBar = 0.0f;
                    if (lowT) maxBar = -ltTot;
                    else if (highT) maxBar = ltTot;
                    else rawBar = ltTot;
                    fbar += maxBar * lnOld;
                    lb.x += maxBar * f;
                    ltOldBar += rawBar;
                    tmbar += rawBar * (ts - vt);
                    const float vtbar = -rawBar * tm;
                    const V2 cbv = mul(tg, vtbar);
                    tbar = tbar + mul(cl0, vtbar);
                    vbB = vbB + cbv;
                    wbB += cross(rB, cbv);
                    rBbar = rBbar + mul(perp_grad(cbv), wB);
                    vbA = vbA - cbv;
                    wbA -= cross(rA, cbv);
                    rAbar = rAbar - mul(perp_grad(cbv), wA);
                    lb.y = ltOldBar;
                }
                if (movA) V[bA] = float4{vbA.x, vbA.y, wbA, va4.w};
                if (movB) V[bB] = float4{vbB.x, vbB.y, wbB, vb4.w};
                a.lamtmp[slot] = lb;
                a.cbar[slot * 3 + 0] = float4{nbar.x, nbar.y, rAbar.x, rAbar.y};
                a.cbar[slot * 3 + 1] = float4{rBbar.x, rBbar.y, tbar.x, tbar.y};
                a.cbar[slot * 3 + 2] = float4{nmbar, tmbar, biasbar, fbar};
            }
            __syncthreads();
            cur = next;
            e = en;
        }
    }
    // Warm start, per slot.  Its deltas do not depend on velocities, so
    // the velocity adjoints here are those after every slot's warm start
    // and before any creation-time term below is added: constraint
    // creation (the restitution bias reads the velocities) precedes the
    // whole island's warm start in the forward step.
    for (int e = lane; e < n; e += kWave) {
        const std::size_t slot = std::size_t(co) + e;
        const float4* vc = vcrec(e);
        if ((__float_as_uint(vc[10].z) >> 8) != 1u) continue;
        const V2 nrm = v2(vc[0]);
        const V2 tg = fwdperp(nrm);
        const V2 rA{vc[3].x, vc[3].y}, rB{vc[3].z, vc[3].w};
        const float lnInit = vc[4].x, ltInit = vc[4].y;
        const float4 ms = vc[8];
        const float mA = ms.x, iA = ms.y, mB = ms.z, iB = ms.w;
        const int bA = __float_as_int(vc[2].w), bB = __float_as_int(vc[5].z);
        float2 lb = a.lamtmp[slot];
        if (c.warmStart) {
            const float4 zero{0.0f, 0.0f, 0.0f, 0.0f};
            const float4 va4 = (mA != 0.0f || iA != 0.0f) ? V[bA] : zero;
            const float4 vb4 = (mB != 0.0f || iB != 0.0f) ? V[bB] : zero;
            const V2 vbA = v2(va4), vbB = v2(vb4);
            const float wbA = va4.z, wbB = vb4.z;
            const float4 c0 = a.cbar[slot * 3 + 0], c1 = a.cbar[slot * 3 + 1];
            V2 nbar{c0.x, c0.y}, rAbar{c0.z, c0.w}, rBbar{c1.x, c1.y}, tbar{c1.z, c1.w};
            const V2 P = mul(lnInit, nrm) + mul(ltInit, tg);
            const V2 Pbar = mul(mB, vbB) - mul(mA, vbA) + mul(revperp(rA), -iA * wbA) + mul(revperp(rB), iB * wbB);
            rAbar = rAbar + mul(perp_grad(P), -iA * wbA);
            rBbar = rBbar + mul(perp_grad(P), iB * wbB);
            lb.x += dot(Pbar, nrm);
            lb.y += dot(Pbar, tg);
            nbar = nbar + mul(Pbar, lnInit);
            tbar = tbar + mul(Pbar, ltInit);
            a.cbar[slot * 3 + 0] = float4{nbar.x, nbar.y, rAbar.x, rAbar.y};
            a.cbar[slot * 3 + 1] = float4{rBbar.x, rBbar.y, tbar.x, tbar.y};
        }
        // Impulses as carried from the previous step (dtRatio scaling is
        // part of the record: warm start uses them as stored); nothing
        // for a contact created before this step's solve.
        const std::uint32_t id = __float_as_uint(vc[10].y);
        const bool fresh = (t.cmap[co + int(id)] & prx::kCarryFresh) != 0u;
        a.lambar[co + int(id)] = fresh ? float4{0.0f, 0.0f, 0.0f, 0.0f} : float4{lb.x, lb.y, lnInit, ltInit};
    }
    __syncthreads();
    // Constraint creation, round by round (its terms add to the bodies').
    int slots = 0, biased = 0;
    for (int r = 0; r < rounds; ++r) {
        const int pos = start[r] + lane;
        const int e = pos < start[r + 1] ? order[pos] : -1;
        if (e >= 0 && (__float_as_uint(vcrec(e)[10].z) >> 8) == 1u) {
            const std::size_t slot = std::size_t(co) + e;
            const float4* vc = vcrec(e);
            const std::uint32_t type = __float_as_uint(vc[10].z) & 0xffu;
            const V2 nrm = v2(vc[0]);
            const V2 tg = fwdperp(nrm);
            const V2 rA{vc[3].x, vc[3].y}, rB{vc[3].z, vc[3].w};
            const float nm = vc[4].z, tm = vc[4].w;
            const float4 ms = vc[8];
            const float mA = ms.x, iA = ms.y, mB = ms.z, iB = ms.w;
            const int bA = __float_as_int(vc[2].w), bB = __float_as_int(vc[5].z);
            const bool movA = mA != 0.0f || iA != 0.0f, movB = mB != 0.0f || iB != 0.0f || V[bB].w != 0.0f;
            const float4 c0 = a.cbar[slot * 3 + 0], c1 = a.cbar[slot * 3 + 1], c2 = a.cbar[slot * 3 + 2];
            V2 nbar{c0.x, c0.y}, rAbar{c0.z, c0.w}, rBbar{c1.x, c1.y}, tbar{c1.z, c1.w};
            const float nmbar = c2.x, tmbar = c2.y, biasbar = c2.z, fbarC = c2.w;
            // Effective masses (VelocityConstraint.cpp:136-185).
            {
                const float cnA = cross(rA, nrm), cnB = cross(rB, nrm);
                const float K = mA + mB + iA * cnA * cnA + iB * cnB * cnB;
                if (K > 0.0f) {
                    const float Kbar = -nmbar * nm * nm;
                    const float gA = 2.0f * iA * cnA * Kbar, gB = 2.0f * iB * cnB * Kbar;
                    rAbar = rAbar + mul(perp_grad(nrm), gA);
                    nbar = nbar + mul(revperp(rA), gA);
                    rBbar = rBbar + mul(perp_grad(nrm), gB);
                    nbar = nbar + mul(revperp(rB), gB);
                }
                const float ctA = cross(rA, tg), ctB = cross(rB, tg);
                const float Kt = mA + mB + iA * ctA * ctA + iB * ctB * ctB;
                if (Kt > 0.0f) {
                    const float Kbar = -tmbar * tm * tm;
                    const float gA = 2.0f * iA * ctA * Kbar, gB = 2.0f * iB * ctB * Kbar;
                    rAbar = rAbar + mul(perp_grad(tg), gA);
                    tbar = tbar + mul(revperp(rA), gA);
                    rBbar = rBbar + mul(perp_grad(tg), gB);
                    tbar = tbar + mul(revperp(rB), gB);
                }
            }
            // Restitution bias from the closing speed at creation.
            const float vn0 = vc[10].x;
            const float rest = vc[5].w;
            const float4 vA0 = vc[12], vB0 = vc[13];
            V2 dvA{0.0f, 0.0f}, dvB{0.0f, 0.0f};
            float dwA = 0.0f, dwB = 0.0f;
            ++slots;
            if (vn0 < -c.velocityThreshold) {
                ++biased;
                const float ebarC = -vn0 * biasbar;
                const float vn0bar = -rest * biasbar;
                const V2 cl0 = (V2{vB0.x, vB0.y} + mul(revperp(rB), vB0.z)) - (V2{vA0.x, vA0.y} + mul(revperp(rA), vA0.z));
                const V2 cbv = mul(nrm, vn0bar);
                nbar = nbar + mul(cl0, vn0bar);
                dvB = cbv;
                dwB = cross(rB, cbv);
                rBbar = rBbar + mul(perp_grad(cbv), vB0.z);
                dvA = -cbv;
                dwA = -cross(rA, cbv);
                rAbar = rAbar - mul(perp_grad(cbv), vA0.z);
                // Restitution = max(eA, eB), ties to B (Contact.hpp:66-69).
                const int sA = __float_as_int(vc[11].y), sB = __float_as_int(vc[11].z);
                const float eA = d.shape_f[sA].z, eB = d.shape_f[sB].z;
                atomicAdd(a.ebar + ((eA > eB) ? sA : sB), ebarC);
            }
            // Friction = sqrt(fA fB) (Contact.hpp:57-60).
            {
                const int sA = __float_as_int(vc[11].y), sB = __float_as_int(vc[11].z);
                const float fA = d.shape_f[sA].y, fB = d.shape_f[sB].y;
                const float fm = vc[0].z;
                if (fm > 0.0f) {
                    atomicAdd(a.fbar + sA, fbarC * fB / (2.0f * fm));
                    atomicAdd(a.fbar + sB, fbarC * fA / (2.0f * fm));
                }
            }
            if (movA) add_body(V + bA, dvA, dwA);
            if (movB) add_body(V + bB, dvB, dwB);
            // Geometry (WorldManifold.cpp:37-130): tangent from the normal,
            // then the normal and points from the positions.
            nbar.x += -tbar.y;
            nbar.y += tbar.x;
            const float4 pos4 = vc[9];
            const float rAd = vc[10].w, rBd = vc[11].x;
            if (type == 1u) {
                const V2 dd = V2{pos4.z - pos4.x, pos4.w - pos4.y};
                const float L = __builtin_sqrtf(magsq(dd));
                if (L > 0.0f) {
                    const float k = 0.5f * (rAd - rBd);
                    V2 dbar = mul(rAbar - rBbar, 0.5f);
                    const V2 ntot = nbar + mul(rAbar + rBbar, k);
                    const float nn = dot(nrm, ntot);
                    dbar = dbar + mul(ntot - mul(nrm, nn), 1.0f / L);
                    if (movA) add_body(X + bA, -dbar, 0.0f);
                    if (movB) add_body(X + bB, dbar, 0.0f);
                }
            } else if (type == 2u) {
                // relB = ((rA - dd) - rB) / 2 n with dd = dot(cB - plane, n);
                // the normal and plane belong to the static body.
                const float ddbar = -0.5f * dot(rBbar, nrm);
                if (movB) add_body(X + bB, mul(nrm, ddbar), 0.0f);
            }
        }
        __syncthreads();
    }
    // Velocity integration, reversed (damping factors; caps not active).
    for (int b = lane; b < nb; b += kWave) {
        const int gb = bo + b;
        float4 v = V[b];
        if (t.inisl[gb] && (d.bflags[gb] & prx::kAccelerable)) {
            const float2 dm = d.damp[gb];
            const float fl = 1.0f / (1.0f + c.dt * dm.x);
            const float fa = 1.0f / (1.0f + c.dt * dm.y);
            v.x *= fl;
            v.y *= fl;
            v.z *= fa;
        }
        a.vbar[gb] = v;
        if constexpr (kLds) a.xbar[gb] = X[b];
    }
    if (unmodelled) *a.status = 1;
    add_diag(a.diag, 0, slots);
    add_diag(a.diag, 1, biased);
    add_diag(a.diag, 2, posUpdates);
    add_diag(a.diag, 3, velUpdates);
}

// ---------------------------------------------------------------------------
// General form: any manifold type and point count, revolute joints, bodies
// with local centres.  The active set is held fixed as recorded; each solver
// update is reversed by its vector-Jacobian product, which the wave computes
// from the update's dual copy (adjoint_dual.hpp): lane i evaluates the copy
// with input i seeded and returns sum_j ybar_j d y_j / d x_i.

template <int N, int M, class F>
__device__ __forceinline__ float lane_vjp(const float (&x)[N], const float (&ybar)[M], F f) {
    const int lane = int(threadIdx.x) & (kWave - 1);
    dl::D in[N];
#pragma unroll
    for (int i = 0; i < N; ++i) in[i] = dl::D{x[i], (i == lane) ? 1.0f : 0.0f};
    dl::D out[M];
    f(in, out);
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < M; ++j) s += ybar[j] * out[j].d;
    return (lane < N) ? s : 0.0f;
}

// Velocity-constraint values a contact's updates read, in the order of the
// creation outputs (kAdjFields): normal x, y; friction; point 0 relA, relB,
// ni, ti, normal mass, tangent mass, bias; point 1 the same; K00, K11, K01,
// M00, M11, M01.
__device__ __forceinline__ void vc_fields(const float4* v, float (&f)[27]) {
    f[0] = v[0].x; f[1] = v[0].y; f[2] = v[0].z;
    f[3] = v[3].x; f[4] = v[3].y; f[5] = v[3].z; f[6] = v[3].w;
    f[7] = v[4].x; f[8] = v[4].y; f[9] = v[4].z; f[10] = v[4].w; f[11] = v[5].x;
    f[12] = v[6].x; f[13] = v[6].y; f[14] = v[6].z; f[15] = v[6].w;
    f[16] = v[7].x; f[17] = v[7].y; f[18] = v[7].z; f[19] = v[7].w; f[20] = v[5].y;
    f[21] = v[1].x; f[22] = v[1].y; f[23] = v[1].z; f[24] = v[2].x; f[25] = v[2].y; f[26] = v[2].z;
}
__device__ __forceinline__ dl::Vcd vcd_from(const dl::D* f, const float4* v) {
    dl::Vcd vc;
    vc.normal = dl::V{f[0], f[1]};
    vc.friction = f[2];
    vc.tangentSpeed = v[0].w;
    vc.n = __float_as_uint(v[1].w);
    vc.p[0] = dl::VcPointD{dl::V{f[3], f[4]}, dl::V{f[5], f[6]}, f[7], f[8], f[9], f[10], f[11]};
    vc.p[1] = dl::VcPointD{dl::V{f[12], f[13]}, dl::V{f[14], f[15]}, f[16], f[17], f[18], f[19], f[20]};
    vc.K00 = f[21]; vc.K11 = f[22]; vc.K01 = f[23]; vc.M00 = f[24]; vc.M11 = f[25]; vc.M01 = f[26];
    return vc;
}

// Joint record values its updates read (kAdjJointFields): rA, rB; exx, eyx,
// ezx, eyy, ezy, ezz; angular mass; impulses x, y, z, motor; max impulse.
__device__ __forceinline__ void jc_fields(const float4* u, float (&f)[16]) {
    f[0] = u[0].x; f[1] = u[0].y; f[2] = u[0].z; f[3] = u[0].w;
    f[4] = u[1].x; f[5] = u[1].y; f[6] = u[1].z; f[7] = u[1].w;
    f[8] = u[2].x; f[9] = u[2].y; f[10] = u[2].z;
    f[11] = u[3].x; f[12] = u[3].y; f[13] = u[3].z; f[14] = u[3].w;
    f[15] = u[5].y;
}
__device__ __forceinline__ dl::Jd jd_from(const dl::D* f) {
    dl::Jd j;
    j.rA = dl::V{f[0], f[1]};
    j.rB = dl::V{f[2], f[3]};
    j.exx = f[4]; j.eyx = f[5]; j.ezx = f[6]; j.eyy = f[7]; j.ezy = f[8]; j.ezz = f[9];
    j.angularMass = f[10];
    j.ix = f[11]; j.iy = f[12]; j.iz = f[13]; j.motorImp = f[14];
    j.maxImpulse = f[15];
    return j;
}

__device__ __forceinline__ void load3(const float4& v, float* o) {
    o[0] = v.x;
    o[1] = v.y;
    o[2] = v.z;
}
__device__ __forceinline__ void load4(const float4& v, float* o) {
    o[0] = v.x;
    o[1] = v.y;
    o[2] = v.z;
    o[3] = v.w;
}
// Lane k < 3 of a body's three adjoint components (x, y, angle).
__device__ __forceinline__ float& comp(float4& v, int k) { return k == 0 ? v.x : (k == 1 ? v.y : v.z); }

// kAdjGroups groups of kAdjWidth wavefronts per world: a group reverses the
// rounds (kAdjWidth updates each) of its own iterations, the iterations started
// the plan's period apart.  A chain of 32 joints has 32 rounds an iteration
// but a period of a few, so its eight iterations run nearly side by side.  An
// update's record is at most 64 floats: lane i reads float i two rounds ahead
// (the tape comes from HBM) and the wavefront passes it through its stage in
// LDS.  kLds: the body adjoints and the two round plans (velocity sweeps run
// joints then contacts, position sweeps contacts then joints) in LDS, 36 bytes
// a body and 20 a contact slot or joint, else in global memory.  Bound by the
// instructions of the dual update, one round after another: 512 chain worlds
// 0.45 -> 0.32 ms a step, 96 piles 0.21 -> 0.15 ms, against one wavefront
// walking all updates.  Four wavefronts a SIMD (128 registers) keep two worlds
// on a CU; with the 145 registers it would take, one (0.53 ms for the chains).
// 4 x 1 and 8 x 1 wavefronts: chains 0.33 and 0.31, piles 0.21 and 0.21 ms.
constexpr int kAdjGroups = 4, kAdjWidth = 2;
constexpr int kAdjWaves = kAdjGroups * kAdjWidth;
constexpr int kAdjThreads = kAdjWaves * kWave;
constexpr int kJointItem = 1 << 30;

template <bool kLds>
__global__ __launch_bounds__(kAdjThreads)
__attribute__((amdgpu_waves_per_eu(4))) void k_adjoint_general(DeviceState d, Tape t, AdjState a, StepParams c) {
    __shared__ float4 s_stage[kAdjWaves][kWave / 4];
    __shared__ RoundPlan s_plan[2];
    const int w = int(blockIdx.x);
    const int tid = int(threadIdx.x);
    const int lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const WorldHeader H = d.hdr[w];
    const int bo = H.body_off, co = H.contact_off, nb = H.nbodies, cap = H.contact_cap, jo = H.joint_off;
    const int nisl = t.nisl[w];
    const int4* isl = t.isl + bo + w;
    const int2* islj = t.islj + bo + w;
    const int nslots = nisl > 0 ? isl[nisl - 1].y : 0;
    const int njslots = nisl > 0 ? islj[nisl - 1].y : 0;
    float4* const xbar = kLds ? g_smem : a.xbar + bo;
    float4* const vbar = kLds ? g_smem + nb : a.vbar + bo;
    const int items = nslots + njslots, room = cap + H.njoints;
    int* const plan = a.plan + std::size_t(co + jo) * prx::kAdjPlanInts;
    int* const last = kLds ? reinterpret_cast<int*>(g_smem + 2 * nb) : d.s_stack + 2 * bo;
    int* const orderV = kLds ? reinterpret_cast<int*>(g_smem + 2 * nb) + nb : plan;
    int* const startV = orderV + room;
    int* const orderP = startV + room + 1;
    int* const startP = orderP + room;
    int* const iters = startP + room + 1;  // of a contact's or (behind them) a joint's island
    int* const lvl = plan + 6 * room + 2;
    if constexpr (kLds) {
        for (int b = tid; b < nb; b += kAdjThreads) {
            xbar[b] = a.xbar[bo + b];
            vbar[b] = a.vbar[bo + b];
        }
    }
    auto vcrec = [&](int e) { return t.vc + (std::size_t(co) + std::size_t(e)) * prx::kTapeVc; };
    auto jcrec = [&](int e) { return t.jc + (std::size_t(jo) + std::size_t(e)) * prx::kTapeJc; };

    // Impulse adjoints carried in from the next step.  Contacts: by pool id,
    // each of the next step's points to the point of this step its impulses
    // came from in the manifold update after the solve (the tape's carry
    // map: by ContactFeature, else the nearest point; two points may share
    // one source).  Joints: by joint.
    for (int e = tid; e < nslots; e += kAdjThreads) {
        const float4* vc = vcrec(e);
        const std::uint32_t id = __float_as_uint(vc[10].y);
        const float4 lb = a.lamc[(std::size_t(co) + id) * 2];
        const std::uint32_t cm = t.cmap[std::size_t(co) + id];
        const std::uint32_t nnext = (cm >> 8) & 0xfu;
        const float bn[2] = {lb.x, lb.z}, bt[2] = {lb.y, lb.w};
        float r[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (std::uint32_t j = 0; j < 2; ++j) {
            const std::uint32_t k = (cm >> (4 * j)) & 0xfu;
            if (j < nnext && k < 2u) {
                r[2 * k] += bn[j];
                r[2 * k + 1] += bt[j];
            }
        }
        a.lam4[std::size_t(co) + e] = float4{r[0], r[1], r[2], r[3]};
        float* fl = a.fld + (std::size_t(co) + e) * prx::kAdjFields;
        for (int k = 0; k < prx::kAdjFields; ++k) fl[k] = 0.0f;
    }
    for (int e = tid; e < njslots; e += kAdjThreads) {
        const int jg = __float_as_int(jcrec(e)[7].w);
        a.jlam[std::size_t(jo) + e] = a.jcarry[jg];
        float* fl = a.jfld + (std::size_t(jo) + e) * prx::kAdjJointFields;
        for (int k = 0; k < prx::kAdjJointFields; ++k) fl[k] = 0.0f;
    }
    __syncthreads();
    for (int i = tid; i < cap; i += kAdjThreads) {
        a.lamc[(std::size_t(co) + i) * 2] = float4{0.0f, 0.0f, 0.0f, 0.0f};
        a.lamc[(std::size_t(co) + i) * 2 + 1] = float4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    __syncthreads();

    for (int is = tid; is < nisl; is += kAdjThreads) {
        const int4 rng = isl[is];
        const int2 jr = islj[is];
        for (int e = rng.x; e < rng.y; ++e) iters[e] = rng.z | (rng.w << 16);
        for (int e = jr.x; e < jr.y; ++e) iters[nslots + e] = rng.z | (rng.w << 16);
    }
    // Item k of the velocity (position) order: the world's joints (contacts),
    // then the others; islands share no moving body, so their order among
    // one another is free.
    auto item = [&](int k, bool position) {
        const int first = position ? nslots : njslots;
        const bool contact = (k < first) == position;
        return contact ? (position ? k : k - first) : ((position ? k - first : k) | kJointItem);
    };
    auto moving = [&](int it) {
        if (it & kJointItem) {
            const float4* u = jcrec(it & ~kJointItem);
            const float4 ms = u[4];
            return int2{(ms.x != 0.0f || ms.y != 0.0f) ? __float_as_int(u[5].z) : -1,
                        (ms.z != 0.0f || ms.w != 0.0f) ? __float_as_int(u[5].w) : -1};
        }
        const float4* vc = vcrec(it);
        const float4 ms = vc[8];
        return int2{(ms.x != 0.0f || ms.y != 0.0f) ? __float_as_int(vc[2].w) : -1,
                    (ms.z != 0.0f || ms.w != 0.0f) ? __float_as_int(vc[5].z) : -1};
    };
    if (wave == 0) {
        const RoundPlan pv = plan_rounds(items, nb, kAdjWidth, lane, [&](int k) { return moving(item(k, false)); }, last,
                                         lvl, orderV, startV);
        const RoundPlan pp = plan_rounds(items, nb, kAdjWidth, lane, [&](int k) { return moving(item(k, true)); }, last,
                                         lvl, orderP, startP);
        if (lane == 0) {
            s_plan[0] = pv;
            s_plan[1] = pp;
        }
    }
    __syncthreads();
    float* const stage = reinterpret_cast<float*>(&s_stage[wave][0]);
    const float4* const rec = &s_stage[wave][0];
    // The wavefront's own reads, then writes, of a body's adjoints: ordered
    // within the wavefront (no other touches these bodies in the round).
    auto own = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
    // The groups' first wavefronts on different SIMDs: most rounds of a chain
    // hold one update.
    const int group = wave % kAdjGroups, sub = wave / kAdjGroups;
    auto sweeps = [&](bool position, auto fetch, auto reverse) {
        const int rounds = __builtin_amdgcn_readfirstlane(s_plan[position].rounds);
        const int iterations = max_iterations(isl, nisl, lane, position);
        if (rounds == 0 || iterations == 0) return;
        const int* const start = position ? startP : startV;
        const int* const order = position ? orderP : orderV;
        // A group ends an iteration before it starts its next.
        const int period = max(__builtin_amdgcn_readfirstlane(s_plan[position].period),
                               (rounds + kAdjGroups - 1) / kAdjGroups);
        struct At {
            int code;  // -1: none
            float f;
        };
        // The group's place at the tick read ahead, counted from the last
        // round of the last iteration.
        int back = -group * period, done = group;
        auto ahead = [&] {
            At n{-1, 0.0f};
            if (back >= 0 && back < rounds && done < iterations) {
                const int r = rounds - 1 - back, it = iterations - 1 - done;
                const int pos = start[r] + sub;
                if (pos < start[r + 1]) {
                    const int code = item(order[pos], position);
                    const int ran = iters[(code & kJointItem) ? nslots + (code & ~kJointItem) : code];
                    if (it < (position ? ran >> 16 : ran & 0xffff)) {
                        n.code = __builtin_amdgcn_readfirstlane(code);
                        n.f = fetch(n.code, it);
                    }
                }
            }
            if (++back == kAdjGroups * period) {
                back = 0;
                done += kAdjGroups;
            }
            return n;
        };
        At cur = ahead(), next = ahead();
        for (int tick = rounds + (iterations - 1) * period; tick > 0; --tick) {
            if (cur.code >= 0) stage[lane] = cur.f;
            const At after = ahead();
            own();
            if (cur.code >= 0) reverse(cur.code);
            __syncthreads();
            cur = next;
            next = after;
        }
    };
    const float4 zero{0.0f, 0.0f, 0.0f, 0.0f};
    auto set3 = [&](float4* bar, int bA, bool movA, int bB, bool movB, float r) {
        if (lane < 3 && movA) comp(bar[bA], lane) = r;
        else if (lane >= 3 && lane < 6 && movB) comp(bar[bB], lane - 3) = r;
    };

    // Position sweeps, reversed: per iteration the joints (after the
    // contacts in the forward pass), then the contacts, each in reverse.
    int posUpdates = 0;
    sweeps(true,
        [&](int code, int it) {
            if (code & kJointItem) {
                const int e = code & ~kJointItem;
                const float* u = &jcrec(e)[0].x;
                const float* q = &t.jngs[((std::size_t(jo) + e) * std::size_t(t.itP) + it) * 2].x;
                constexpr int kU = 4 * prx::kJcStride;
                return lane < kU ? u[lane] : (lane < kU + 8 ? q[lane - kU] : 0.0f);
            }
            const float* pcr = &vcrec(code)[17].x;
            const float* q = &t.ngs[((std::size_t(co) + code) * std::size_t(t.itP) + it) * 2].x;
            constexpr int kU = 4 * prx::kPcStride;
            return lane < kU ? pcr[lane] : (lane < kU + 8 ? q[lane - kU] : 0.0f);
        },
        [&](int code) {
            if (code & kJointItem) {
                const float4* u = rec;
                const int bA = __float_as_int(u[5].z), bB = __float_as_int(u[5].w);
                const bool movA = u[4].x != 0.0f || u[4].y != 0.0f, movB = u[4].z != 0.0f || u[4].w != 0.0f;
                const float4* g = rec + prx::kJcStride;
                float x[6], yb[6];
                load3(g[0], x);
                load3(g[1], x + 3);
                load3(movA ? xbar[bA] : zero, yb);
                load3(movB ? xbar[bB] : zero, yb + 3);
                const float r = lane_vjp<6, 6>(x, yb, [&](dl::D* in, dl::D* out) {
                    dl::joint_solve_position(u, in, c);
                    for (int k = 0; k < 6; ++k) out[k] = in[k];
                });
                own();
                set3(xbar, bA, movA, bB, movB, r);
                return;
            }
            const std::size_t slot = std::size_t(co) + code;
            const Pc pc = load_pc(rec);
            const bool movA = pc.A.invMass != 0.0f || pc.A.invRotI != 0.0f, movB = pc.B.invMass != 0.0f || pc.B.invRotI != 0.0f;
            const float4* g = rec + prx::kPcStride;
            float* const sum = a.fld + slot * prx::kAdjFields + 28 + (lane - 6);
            const float before = (lane >= 6 && lane < 10) ? *sum : 0.0f;
            // Positions before the update, then the manifold's local
            // points (their adjoints collect for the constraint creation).
            float x[10], yb[6];
            load3(g[0], x);
            load3(g[1], x + 3);
            x[6] = pc.m.p[0].lp.x;
            x[7] = pc.m.p[0].lp.y;
            x[8] = pc.m.p[1].lp.x;
            x[9] = pc.m.p[1].lp.y;
            load3(movA ? xbar[pc.bA] : zero, yb);
            load3(movB ? xbar[pc.bB] : zero, yb + 3);
            const float r = lane_vjp<10, 6>(x, yb, [&](dl::D* in, dl::D* out) {
                const dl::V lpd[2] = {dl::V{in[6], in[7]}, dl::V{in[8], in[9]}};
                dl::solve_pc(pc.m, pc.totalRadius, pc.A, pc.B, in, c, lpd);
                for (int k = 0; k < 6; ++k) out[k] = in[k];
            });
            own();
            set3(xbar, pc.bA, movA, pc.bB, movB, r);
            if (lane >= 6 && lane < 10) *sum = before + r;
            ++posUpdates;
        });
    __syncthreads();
    // Position integration, reversed: x1 = x0 + h v.
    for (int b = tid; b < nb; b += kAdjThreads) {
        if (!t.inisl[bo + b]) continue;
        const float4 xb = xbar[b];
        add_body(vbar + b, V2{c.dt * xb.x, c.dt * xb.y}, c.dt * xb.z);
    }
    __syncthreads();

    // Velocity sweeps, reversed: per iteration the contacts, then the
    // joints (solved first in the forward pass), each in reverse.
    int velUpdates = 0;
    sweeps(false,
        [&](int code, int it) {
            if (code & kJointItem) {
                const int e = code & ~kJointItem;
                const float* u = &jcrec(e)[0].x;
                const float* q = &t.jgs[((std::size_t(jo) + e) * std::size_t(t.itV) + it) * 3].x;
                constexpr int kU = 4 * prx::kJcStride;
                return lane < kU ? u[lane] : (lane < kU + 12 ? q[lane - kU] : 0.0f);
            }
            const float* v = &vcrec(code)[0].x;
            const float* q = &t.gs[((std::size_t(co) + code) * std::size_t(t.itV) + it) * 3].x;
            constexpr int kU = 4 * prx::kVcStride;
            return lane < kU ? v[lane] : (lane < kU + 12 ? q[lane - kU] : 0.0f);
        },
        [&](int code) {
            if (code & kJointItem) {
                const std::size_t js = std::size_t(jo) + (code & ~kJointItem);
                const float4* u = rec;
                const int bA = __float_as_int(u[5].z), bB = __float_as_int(u[5].w);
                const bool movA = u[4].x != 0.0f || u[4].y != 0.0f, movB = u[4].z != 0.0f || u[4].w != 0.0f;
                const float4* g = rec + prx::kJcStride;
                float f[16];
                jc_fields(u, f);
                float x[22], yb[10];
                load3(g[0], x);
                load3(g[1], x + 3);
                load4(g[2], x + 6);
                constexpr int kJMap[12] = {0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 15};
                const bool summed = lane >= 10 && lane < 22;
                float* const sum = a.jfld + js * prx::kAdjJointFields + (lane == 21 ? 15 : lane - 10);  // kJMap[lane - 10]
                const float before = summed ? *sum : 0.0f;
#pragma unroll
                for (int k = 0; k < 12; ++k) x[10 + k] = f[kJMap[k]];
                load3(movA ? vbar[bA] : zero, yb);
                load3(movB ? vbar[bB] : zero, yb + 3);
                load4(a.jlam[js], yb + 6);
                const float r = lane_vjp<22, 10>(x, yb, [&](dl::D* in, dl::D* out) {
                    dl::D fd[16];
                    for (int k = 0; k < 16; ++k) fd[k] = dl::cst(f[k]);
#pragma unroll
                    for (int k = 0; k < 12; ++k) fd[kJMap[k]] = in[10 + k];
                    fd[11] = in[6];
                    fd[12] = in[7];
                    fd[13] = in[8];
                    fd[14] = in[9];
                    dl::Jd j = jd_from(fd);
                    dl::D va[3] = {in[0], in[1], in[2]}, vb[3] = {in[3], in[4], in[5]};
                    dl::joint_solve_velocity(j, u, va, vb);
                    for (int k = 0; k < 3; ++k) {
                        out[k] = va[k];
                        out[3 + k] = vb[k];
                    }
                    out[6] = j.ix;
                    out[7] = j.iy;
                    out[8] = j.iz;
                    out[9] = j.motorImp;
                });
                own();
                set3(vbar, bA, movA, bB, movB, r);
                if (lane >= 6 && lane < 10) (&a.jlam[js].x)[lane - 6] = r;
                else if (summed) *sum = before + r;
                return;
            }
            const std::size_t slot = std::size_t(co) + code;
            const float4* vc = rec;
            const int bA = __float_as_int(vc[2].w), bB = __float_as_int(vc[5].z);
            const BodyC A{vc[8].x, vc[8].y, V2{0, 0}}, B{vc[8].z, vc[8].w, V2{0, 0}};
            const bool movA = A.invMass != 0.0f || A.invRotI != 0.0f, movB = B.invMass != 0.0f || B.invRotI != 0.0f;
            const float4* g = rec + prx::kVcStride;
            float x[33], yb[10];
            load3(g[0], x);
            load3(g[1], x + 3);
            load4(g[2], x + 6);
            float f[27];
            vc_fields(vc, f);
            // Fields the update reads (creation-output indices).
            constexpr int kMap[23] = {0, 1, 2, 3, 4, 5, 6, 9, 10, 11, 12, 13, 14, 15, 18, 19, 20, 21, 22, 23, 24, 25, 26};
            const bool summed = lane >= 10 && lane < 33;
            // kMap[lane - 10]: the impulses' places (7, 8 and 16, 17) are skipped.
            float* const sum = a.fld + slot * prx::kAdjFields + (lane - 10 + (lane >= 17 ? 2 : 0) + (lane >= 24 ? 2 : 0));
            const float before = summed ? *sum : 0.0f;
#pragma unroll
            for (int k = 0; k < 23; ++k) x[10 + k] = f[kMap[k]];
            load3(movA ? vbar[bA] : zero, yb);
            load3(movB ? vbar[bB] : zero, yb + 3);
            load4(a.lam4[slot], yb + 6);
            const float r = lane_vjp<33, 10>(x, yb, [&](dl::D* in, dl::D* out) {
                dl::D fd[27];
                for (int k = 0; k < 27; ++k) fd[k] = dl::cst(f[k]);
#pragma unroll
                for (int k = 0; k < 23; ++k) fd[kMap[k]] = in[10 + k];
                fd[7] = in[6];
                fd[8] = in[7];
                fd[16] = in[8];
                fd[17] = in[9];
                dl::Vcd v = vcd_from(fd, vc);
                dl::D va[3] = {in[0], in[1], in[2]}, vb[3] = {in[3], in[4], in[5]};
                dl::solve_velocity(v, A, B, va, vb);
                for (int k = 0; k < 3; ++k) {
                    out[k] = va[k];
                    out[3 + k] = vb[k];
                }
                out[6] = v.p[0].ni;
                out[7] = v.p[0].ti;
                out[8] = v.p[1].ni;
                out[9] = v.p[1].ti;
            });
            own();
            set3(vbar, bA, movA, bB, movB, r);
            if (lane >= 6 && lane < 10) (&a.lam4[slot].x)[lane - 6] = r;
            else if (summed) *sum = before + r;
            ++velUpdates;
        });
    // What follows is independent per joint and per contact but for the sums
    // at the bodies.
    // Joint warm start, reversed (after the contacts' in the forward
    // pass; linear in the velocities, so their values do not enter).
    for (int e = wave; e < njslots; e += kAdjWaves) {
        const std::size_t js = std::size_t(jo) + e;
        const float4* u = jcrec(e);
        const int bA = __float_as_int(u[5].z), bB = __float_as_int(u[5].w);
        if (c.warmStart) {
            float f[16];
            jc_fields(u, f);
            float x[14] = {0, 0, 0, 0, 0, 0, f[0], f[1], f[2], f[3], f[11], f[12], f[13], f[14]};
            float yb[6];
            load3((u[4].x != 0.0f || u[4].y != 0.0f) ? vbar[bA] : zero, yb);
            load3((u[4].z != 0.0f || u[4].w != 0.0f) ? vbar[bB] : zero, yb + 3);
            const float r = lane_vjp<14, 6>(x, yb, [&](dl::D* in, dl::D* out) {
                dl::D fd[16];
                for (int k = 0; k < 16; ++k) fd[k] = dl::cst(f[k]);
                for (int k = 0; k < 4; ++k) fd[k] = in[6 + k];
                for (int k = 0; k < 4; ++k) fd[11 + k] = in[10 + k];
                const dl::Jd j = jd_from(fd);
                dl::D va[3] = {in[0], in[1], in[2]}, vb[3] = {in[3], in[4], in[5]};
                dl::joint_warm_start(j, u, va, vb);
                for (int k = 0; k < 3; ++k) {
                    out[k] = va[k];
                    out[3 + k] = vb[k];
                }
            });
            own();
            if (lane >= 6 && lane < 10) a.jfld[js * prx::kAdjJointFields + (lane - 6)] += r;
            else if (lane >= 10 && lane < 14) a.jfld[js * prx::kAdjJointFields + 11 + (lane - 10)] += r;
            own();
        }
        // The sweeps started from the set-up's impulses.
        if (lane < 4) a.jfld[js * prx::kAdjJointFields + 11 + lane] += (&a.jlam[js].x)[lane];
        own();
    }
    // Contact warm start, reversed (linear in the velocities).
    for (int e = wave; e < nslots; e += kAdjWaves) {
        const std::size_t slot = std::size_t(co) + e;
        const float4* vc = vcrec(e);
        const int bA = __float_as_int(vc[2].w), bB = __float_as_int(vc[5].z);
        const BodyC A{vc[8].x, vc[8].y, V2{0, 0}}, B{vc[8].z, vc[8].w, V2{0, 0}};
        if (c.warmStart) {
            float f[27];
            vc_fields(vc, f);
            constexpr int kWMap[14] = {0, 1, 3, 4, 5, 6, 7, 8, 12, 13, 14, 15, 16, 17};
            float x[20] = {0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < 14; ++k) x[6 + k] = f[kWMap[k]];
            float yb[6];
            load3((A.invMass != 0.0f || A.invRotI != 0.0f) ? vbar[bA] : zero, yb);
            load3((B.invMass != 0.0f || B.invRotI != 0.0f) ? vbar[bB] : zero, yb + 3);
            const float r = lane_vjp<20, 6>(x, yb, [&](dl::D* in, dl::D* out) {
                dl::D fd[27];
                for (int k = 0; k < 27; ++k) fd[k] = dl::cst(f[k]);
#pragma unroll
                for (int k = 0; k < 14; ++k) fd[kWMap[k]] = in[6 + k];
                const dl::Vcd v = vcd_from(fd, vc);
                dl::D va[3] = {in[0], in[1], in[2]}, vb[3] = {in[3], in[4], in[5]};
                dl::warm_start(v, A, B, va, vb);
                for (int k = 0; k < 3; ++k) {
                    out[k] = va[k];
                    out[3 + k] = vb[k];
                }
            });
            own();
            if (lane >= 6 && lane < 20) a.fld[slot * prx::kAdjFields + kWMap[lane - 6]] += r;
            own();
        }
        // The sweeps started from the warm-start impulses.
        if (lane < 4) {
            constexpr int kImp[4] = {7, 8, 16, 17};
            a.fld[slot * prx::kAdjFields + kImp[lane]] += (&a.lam4[slot].x)[lane];
        }
        own();
    }
    __syncthreads();
    // Joint set-up, reversed: angles, the impulses it started from and
    // the maximum motor torque.
    auto joint_setup = [&](int e) {
        const std::size_t js = std::size_t(jo) + e;
        const float4* u = jcrec(e);
        const int bA = __float_as_int(u[5].z), bB = __float_as_int(u[5].w);
        const int jg = __float_as_int(u[7].w);
        const float4 in8 = u[prx::kJcStride], raw = u[prx::kJcStride + 1];
        float x[7] = {in8.x, in8.y, raw.x, raw.y, raw.z, raw.w, in8.z};
        float yb[16];
        for (int k = 0; k < 16; ++k) yb[k] = a.jfld[js * prx::kAdjJointFields + k];
        const std::uint32_t prevLimit = __float_as_uint(in8.w);
        const float r = lane_vjp<7, 16>(x, yb, [&](dl::D* in, dl::D* out) {
            const dl::Jd j = dl::build_jc(in[0], in[1], in + 2, in[6], u, prevLimit, c);
            out[0] = j.rA.x; out[1] = j.rA.y; out[2] = j.rB.x; out[3] = j.rB.y;
            out[4] = j.exx; out[5] = j.eyx; out[6] = j.ezx; out[7] = j.eyy; out[8] = j.ezy; out[9] = j.ezz;
            out[10] = j.angularMass;
            out[11] = j.ix; out[12] = j.iy; out[13] = j.iz; out[14] = j.motorImp;
            out[15] = j.maxImpulse;
        });
        own();
        if (lane < 2) {
            const bool mov = lane == 0 ? (u[4].x != 0.0f || u[4].y != 0.0f) : (u[4].z != 0.0f || u[4].w != 0.0f);
            a.jfld[js * prx::kAdjJointFields + lane] = r;
            a.jfld[js * prx::kAdjJointFields + 2 + lane] = __int_as_float(mov ? (lane == 0 ? bA : bB) : -1);
        } else if (lane < 6) (&a.jcarry[jg].x)[lane - 2] = r;
        else if (lane == 6) a.tbar[jg] += r;
        own();
    };
    // Contact constraint creation, reversed: positions and velocities at
    // creation, materials, and the manifold impulses it started from.
    auto contact_creation = [&](int e) {
        const std::size_t slot = std::size_t(co) + e;
        const float4* vc = vcrec(e);
        const Pc pc = load_pc(vc + 17);
        const std::uint32_t id = __float_as_uint(vc[10].y);
        const float rA = vc[10].w, rB = vc[11].x;
        float x[22];
        load3(vc[15], x);
        load3(vc[16], x + 3);
        load3(vc[12], x + 6);
        load3(vc[13], x + 9);
        x[12] = vc[0].z;
        x[13] = vc[5].w;
        load4(vc[22], x + 14);
        x[18] = pc.m.p[0].lp.x;
        x[19] = pc.m.p[0].lp.y;
        x[20] = pc.m.p[1].lp.x;
        x[21] = pc.m.p[1].lp.y;
        float yb[27];
        for (int k = 0; k < 27; ++k) yb[k] = a.fld[slot * prx::kAdjFields + k];
        const float r = lane_vjp<22, 27>(x, yb, [&](dl::D* in, dl::D* out) {
            const dl::X xfA = dl::get_xf(in[0], in[1], in[2], pc.A.lc);
            const dl::X xfB = dl::get_xf(in[3], in[4], in[5], pc.B.lc);
            const dl::V lpd[2] = {dl::V{in[18], in[19]}, dl::V{in[20], in[21]}};
            const dl::WMd wm = dl::world_manifold(pc.m, xfA, rA, xfB, rB, lpd);
            const dl::Vcd v = dl::make_vc(wm, in[12], in[13], vc[0].w, pc.A, in, in + 6, pc.B, in + 3, in + 9,
                                          in + 14, c);
            out[0] = v.normal.x; out[1] = v.normal.y; out[2] = v.friction;
            for (int k = 0; k < 2; ++k) {
                const dl::VcPointD& p = v.p[k];
                dl::D* o = out + 3 + 9 * k;
                o[0] = p.relA.x; o[1] = p.relA.y; o[2] = p.relB.x; o[3] = p.relB.y;
                o[4] = p.ni; o[5] = p.ti; o[6] = p.nm; o[7] = p.tm; o[8] = p.bias;
            }
            out[21] = v.K00; out[22] = v.K11; out[23] = v.K01; out[24] = v.M00; out[25] = v.M11; out[26] = v.M01;
        });
        own();
        const bool movA = pc.A.invMass != 0.0f || pc.A.invRotI != 0.0f, movB = pc.B.invMass != 0.0f || pc.B.invRotI != 0.0f;
        float term = r;  // lanes 0-5 positions, 6-11 velocities, 12 friction, 13 restitution
        if (lane >= 14 && lane < 18) {
            // Nothing for a contact created before this step's solve.
            const bool fresh = (t.cmap[std::size_t(co) + id] & prx::kCarryFresh) != 0u;
            (&a.lamc[(std::size_t(co) + id) * 2].x)[lane - 14] = fresh ? 0.0f : r;
            (&a.lamc[(std::size_t(co) + id) * 2 + 1].x)[lane - 14] = (&vc[22].x)[lane - 14];
        } else if (lane >= 18 && lane < 22) {
            a.fld[slot * prx::kAdjFields + 28 + (lane - 18)] += r;
        }
        own();
        // The manifold's local points as made by the update before this
        // step, at the same positions: points the clipping made move
        // with the bodies.
        const std::uint32_t mtype = pc.m.type;
        const float4 cfs = vc[23];
        if (mtype == kFaceA || mtype == kFaceB) {
            const bool faceB = mtype == kFaceB;
            const int sA = __float_as_int(vc[11].y), sB = __float_as_int(vc[11].z);
            const Proxy s0 = shape_proxy(d, faceB ? sB : sA), s1 = shape_proxy(d, faceB ? sA : sB);
            float xm[6], ybm[4];
            load3(vc[15], xm);
            load3(vc[16], xm + 3);
            for (int k = 0; k < 4; ++k) ybm[k] = a.fld[slot * prx::kAdjFields + 28 + k];
            const float rm = lane_vjp<6, 4>(xm, ybm, [&](dl::D* in, dl::D* out) {
                const dl::X xfA = dl::get_xf(in[0], in[1], in[2], pc.A.lc);
                const dl::X xfB = dl::get_xf(in[3], in[4], in[5], pc.B.lc);
                for (std::uint32_t k = 0; k < 2; ++k) {
                    dl::V lp = dl::vc2(pc.m.p[k].lp);
                    if (k < pc.m.n)
                        lp = dl::manifold_local_point(s0, faceB ? xfB : xfA, s1, faceB ? xfA : xfB,
                                                      __float_as_uint(k ? cfs.y : cfs.x), faceB, pc.m.ln,
                                                      pc.m.p[k].lp);
                    out[2 * k] = lp.x;
                    out[2 * k + 1] = lp.y;
                }
            });
            own();
            if (lane < 6) term += rm;
        }
        // The record's sums have been read: its place takes the terms and
        // the moving bodies they go to.
        if (lane < 14) a.fld[slot * prx::kAdjFields + lane] = term;
        else if (lane < 16) a.fld[slot * prx::kAdjFields + lane] = __int_as_float(lane == 14 ? (movA ? pc.bA : -1) : (movB ? pc.bB : -1));
    };
    for (int k = wave; k < items; k += kAdjWaves) {
        const int code = item(k, false);
        if (code & kJointItem) joint_setup(code & ~kJointItem);
        else contact_creation(code);
    }
    __syncthreads();
    // The sums: the bodies' by one wavefront round after round (twelve lanes an
    // item), in one order whatever the wavefronts' timing; the materials' by
    // another, slots in order, a wavefront's additions to one shape's word in
    // the order its atomics take (the same from run to run as measured, but
    // nothing that the hardware promises).
    if (wave == 0) {
        const int l = lane % 12;
        const bool toB = (l % 6) >= 3;
        struct Term {
            float v;
            int b;
        };
        auto term_of = [&](int r) {
            Term n{0.0f, -1};
            const int pos = r >= 0 ? startV[r] + lane / 12 : 0;
            if (r < 0 || lane >= 12 * kAdjWidth || pos >= startV[r + 1]) return n;
            const int code = item(orderV[pos], false);
            if (code & kJointItem) {
                const float* f = a.jfld + (std::size_t(jo) + (code & ~kJointItem)) * prx::kAdjJointFields;
                if (l == 2 || l == 5) n = Term{f[toB ? 1 : 0], __float_as_int(f[toB ? 3 : 2])};
            } else {
                const float* f = a.fld + (std::size_t(co) + code) * prx::kAdjFields;
                n = Term{f[l], __float_as_int(f[toB ? 15 : 14])};
            }
            return n;
        };
        Term cur = term_of(s_plan[0].rounds - 1);
        for (int r = s_plan[0].rounds - 1; r >= 0; --r) {
            const Term next = term_of(r - 1);
            if (cur.b >= 0) comp((l < 6 ? xbar : vbar)[cur.b], l % 3) += cur.v;
            own();
            cur = next;
        }
    } else if (wave == 1) {
        for (int base = nslots - 1; base >= 0; base -= kWave) {
            const int e = base - lane;
            if (e < 0) continue;
            const float4* vc = vcrec(e);
            const float* f = a.fld + (std::size_t(co) + e) * prx::kAdjFields;
            const int sA = __float_as_int(vc[11].y), sB = __float_as_int(vc[11].z);
            // Friction = sqrt(fA fB) (Contact.hpp:57-60).
            const float4 mA = d.shape_f[sA], mB = d.shape_f[sB];
            const float fm = vc[0].z;
            if (fm > 0.0f) {
                atomicAdd(a.fbar + sA, f[12] * mB.y / (2.0f * fm));
                atomicAdd(a.fbar + sB, f[12] * mA.y / (2.0f * fm));
            }
            // Restitution = max(eA, eB), ties to B (Contact.hpp:66-69).
            atomicAdd(a.ebar + ((mA.z > mB.z) ? sA : sB), f[13]);
        }
    }
    __syncthreads();
    // Velocity integration, reversed (damping factors; caps not active).
    for (int b = tid; b < nb; b += kAdjThreads) {
        if (!t.inisl[bo + b]) continue;
        const int gb = bo + b;
        if (!(d.bflags[gb] & prx::kAccelerable)) continue;
        const float2 dm = d.damp[gb];
        const float fl = 1.0f / (1.0f + c.dt * dm.x);
        const float fa = 1.0f / (1.0f + c.dt * dm.y);
        float4 v = vbar[b];
        v.x *= fl;
        v.y *= fl;
        v.z *= fa;
        vbar[b] = v;
    }
    // Bodies that do not move carry no adjoint (the reverse updates leave
    // scratch values there, which never reach a moving body: their inverse
    // masses are zero).
    for (int b = tid; b < nb; b += kAdjThreads) {
        const bool moves = (d.bflags[bo + b] & prx::kAccelerable) != 0;
        if (kLds || !moves) {
            a.xbar[bo + b] = moves ? xbar[b] : zero;
            a.vbar[bo + b] = moves ? vbar[b] : zero;
        }
    }
    if (lane == 0) {
        if (wave == 0 && nslots) atomicAdd(a.diag, float(nslots));
        if (posUpdates) atomicAdd(a.diag + 2, float(posUpdates));
        if (velUpdates) atomicAdd(a.diag + 3, float(velUpdates));
    }
}

}  // namespace prxd

namespace {
// The body adjoints and round plans are kept in LDS where the largest world's
// fit the default limit.
constexpr std::size_t kAdjLdsLimit = 60 * 1024;
}  // namespace

extern "C" hipError_t prx_launch_adjoint_general(const prx::DeviceState* d, const prx::Tape* t,
                                                 const prx::AdjState* a, const prx::StepParams* c, int nworlds,
                                                 int maxBodies, int maxSlots, hipStream_t s) {
    const std::size_t lds = std::size_t(maxBodies) * 36 + std::size_t(maxSlots) * 20 + 8;
    const dim3 grid{unsigned(nworlds)}, block(prxd::kAdjThreads);
    if (lds <= kAdjLdsLimit) hipLaunchKernelGGL(prxd::k_adjoint_general<true>, grid, block, lds, s, *d, *t, *a, *c);
    else hipLaunchKernelGGL(prxd::k_adjoint_general<false>, grid, block, 0, s, *d, *t, *a, *c);
    return hipGetLastError();
}

extern "C" hipError_t prx_launch_adjoint_step(const prx::DeviceState* d, const prx::Tape* t, const prx::AdjState* a,
                                              const prx::StepParams* c, int nworlds, int maxBodies, int maxSlots,
                                              hipStream_t s) {
    const std::size_t lds = std::size_t(maxBodies) * 36 + std::size_t(maxSlots) * 12 + 4;
    const dim3 grid{unsigned(nworlds)}, block(64);
    if (lds <= kAdjLdsLimit) hipLaunchKernelGGL(prxd::k_adjoint_step<true>, grid, block, lds, s, *d, *t, *a, *c);
    else hipLaunchKernelGGL(prxd::k_adjoint_step<false>, grid, block, 0, s, *d, *t, *a, *c);
    return hipGetLastError();
}
