// The fused per-world step: one workgroup (one 64-lane wavefront) advances one
// world through PlayRho's regular step, Step(AabbTreeWorld&, const StepConf&)
// (AabbTreeWorld.cpp:2144-2219):
//
//   A  proxy creation for new shapes              CreateProxies        :557-579
//   B  contact destruction (fat AABBs apart)       DestroyContacts      :2290-2331
//   C  narrowphase of flagged contacts             UpdateContacts/Update:2333-2421,2587-2721
//   D  pair finding + contact creation             FindContacts/AddContacts :709-751,2424-2547
//   E  islands (DFS), per-island Gauss-Seidel solve, writeback, sleep
//                                                  SolveReg/SolveRegIslandViaGS :1472-1682
//   F  proxy synchronisation, C and D again        SolveReg             :1532-1557
//   G  (doToi) the TOI phase, in a second kernel   SolveToi             :1752-1831
//
// Lane-parallel phases: proxy AABBs, destruction with stable compaction
// (ballot prefix counts), narrowphase (one lane per contact), candidate pair
// tests, key sort, contact creation, per-body adjacency, synchronisation.
// Order-dependent phases replay the reference order exactly: the island DFS
// (body after body, the wave looking at a body's contacts and joints side by
// side) and the Gauss-Seidel solve (the updates of a round side by side, four
// lanes each, where the level form takes the island; else a lane per island or
// the whole wave for a large one; islands share no dynamic body).
//
// A batch of worlds is one launch: workgroup g steps world schedule[g]
// (largest worlds first), so uneven world sizes balance across the 256 CUs.
#include "step_device.hpp"

namespace prxd {

// At most 168 VGPRs, so that three waves share a SIMD.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void k_step_worlds(DeviceState d,
                                                                                          StepParams c) {
    const int w = d.schedule[blockIdx.x];
    step_world<false>(d, w, c);
}

// The TOI phase (doToi) of every world, after k_step_worlds in the same stream.
__global__ __launch_bounds__(64) void k_toi_worlds(DeviceState d, StepParams c) {
    const int w = d.schedule[blockIdx.x];
    toi_world(d, w, c);
}

// The same step recording its solve for the adjoint (every island swept by
// one lane: coopMin must exceed every island's constraint count).
__global__ __launch_bounds__(64) void k_step_worlds_tape(DeviceState d, StepParams c) {
    const int w = d.schedule[blockIdx.x];
    step_world<true>(d, w, c);
}

}  // namespace prxd

// Host-side launcher (compiled in this translation unit).
extern "C" hipError_t prx_launch_step(const prx::DeviceState* d, const prx::StepParams* c, int first, int count,
                                      hipStream_t stream) {
    prx::DeviceState dd = *d;
    dd.schedule = d->schedule + first;
    hipLaunchKernelGGL(prxd::k_step_worlds, dim3(unsigned(count)), dim3(64), c->ldsBytes, stream, dd, *c);
    if (c->doToi && c->dt != 0.0f) {
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(prxd::k_toi_worlds, dim3(unsigned(count)), dim3(64), 0, stream, dd, *c);
    }
    return hipGetLastError();
}

extern "C" hipError_t prx_launch_step_tape(const prx::DeviceState* d, const prx::StepParams* c, int count,
                                           hipStream_t stream) {
    hipLaunchKernelGGL(prxd::k_step_worlds_tape, dim3(unsigned(count)), dim3(64), c->ldsBytes, stream, *d, *c);
    return hipGetLastError();
}

namespace prxd {

// Body rows of prx_world_get_bodies (both sweep positions, velocity,
// under-active time) and flags, written straight into pinned host memory.  A
// thread per row word keeps the stores coalesced (the link is the bound: 22 MB
// for 500,000 bodies); the loads hit a line each of ten threads shares.
__global__ __launch_bounds__(256) void k_body_view(DeviceState d, float* rows, std::uint32_t* flags, int n) {
    for (int i = int(blockIdx.x * blockDim.x + threadIdx.x); i < 11 * n; i += int(gridDim.x * blockDim.x)) {
        if (i >= 10 * n) {
            flags[i - 10 * n] = d.bflags[i - 10 * n] & 0x7fu;
            continue;
        }
        const int b = i / 10, f = i - 10 * b;
        const float4* src = f < 3 ? d.pos0 : (f < 6 ? d.pos1 : d.vel);
        rows[i] = reinterpret_cast<const float*>(src + b)[f < 6 ? f % 3 : f - 6];
    }
}

// The worlds' status bits combined and the first world's header, into pinned
// host memory (one workgroup).
__global__ __launch_bounds__(1024) void k_report(DeviceState d, std::uint32_t* out) {
    __shared__ std::uint32_t s_or;
    if (threadIdx.x == 0) s_or = 0u;
    __syncthreads();
    std::uint32_t v = 0u;
    for (int w = int(threadIdx.x); w < d.nworlds; w += int(blockDim.x)) v |= std::uint32_t(d.hdr[w].status);
    if (v) atomicOr(&s_or, v);
    __syncthreads();
    if (threadIdx.x == 0) out[0] = s_or;
    constexpr unsigned kWords = sizeof(prx::WorldHeader) / 4;
    if (threadIdx.x < kWords) out[1 + threadIdx.x] = reinterpret_cast<const std::uint32_t*>(d.hdr)[threadIdx.x];
}

}  // namespace prxd

extern "C" hipError_t prx_launch_body_view(const prx::DeviceState* d, float* rows, std::uint32_t* flags, int n,
                                           hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    const unsigned blocks = unsigned((std::size_t(n) * 11 + 255) / 256);
    hipLaunchKernelGGL(prxd::k_body_view, dim3(blocks < 4096u ? blocks : 4096u), dim3(256), 0, stream, *d, rows, flags, n);
    return hipGetLastError();
}

extern "C" hipError_t prx_launch_report(const prx::DeviceState* d, std::uint32_t* out, hipStream_t stream) {
    hipLaunchKernelGGL(prxd::k_report, dim3(1), dim3(d->nworlds < 256 ? 256u : 1024u), 0, stream, *d, out);
    return hipGetLastError();
}

// Diagnostic: evaluates the device sine/cosine (UnitVec::Get) on n angles.
namespace prxd {
__global__ void k_sincos(const float* in, float* out, int n) {
    const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (i < n) {
        const V2 q = unit_from_angle(in[i]);
        out[2 * i] = q.x;
        out[2 * i + 1] = q.y;
    }
}
}  // namespace prxd

extern "C" int prx_selftest_sincos(const float* angles, float* out, int n) {
    if (n <= 0 || !angles || !out) return 1;
    float* d_in = nullptr;
    float* d_out = nullptr;
    if (hipMalloc(&d_in, sizeof(float) * std::size_t(n)) != hipSuccess) return 5;
    if (hipMalloc(&d_out, 2 * sizeof(float) * std::size_t(n)) != hipSuccess) {
        (void)hipFree(d_in);
        return 5;
    }
    hipError_t e = hipMemcpy(d_in, angles, sizeof(float) * std::size_t(n), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(prxd::k_sincos, dim3(unsigned((n + 255) / 256)), dim3(256), 0, 0, d_in, d_out, n);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(out, d_out, 2 * sizeof(float) * std::size_t(n), hipMemcpyDeviceToHost);
    (void)hipFree(d_in);
    (void)hipFree(d_out);
    return e == hipSuccess ? 0 : 5;
}
