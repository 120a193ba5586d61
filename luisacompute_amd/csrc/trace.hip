// trace.hip -- software trace_closest / trace_any on gfx950 (no ray-tracing hardware on CDNA4).
//
// Replaces the reference's lc_accel_trace_closest / lc_accel_trace_any
// (src/backends/cuda/cuda_builtin/cuda_device_resource.h:1783-1829, OptiX hardware traversal)
// with the observable semantics of the CPU backend's AccelImpl::trace_closest / trace_any
// (src/rust/luisa_compute_backend_impl/src/cpu/accel.rs:449-535); the traversal is that of
// wave_walker.h (one ray per lane) or oct_walker.h (eight lanes per ray, for launches of few rays).
//
// Launch design (wave64): a persistent grid; a wave hands rays to its idle lanes from a pool of
// queue slots it claims in chunks (per-XCD queue segments, below), runs `steps` traversal steps,
// then refills finished lanes, so lanes stay busy while rays of different lengths finish. The queue is the concatenation of up to kMaxBatches ray
// batches (each with its own output buffer and visibility mask); an optional permutation
// (`order`) makes lanes fetch rays in sorted order. The ray count is a kernel argument, or is
// read from device memory (`count_ptr`) for launches whose queue length is produced on the GPU.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cstdint>
#include <map>
#include <mutex>

#include "lc_hip_bvh.h"
#include "lc_hip_internal.h"
#include "oct_walker.h"
#include "wave_walker.h"

// Working memory of lc_hip_accel_trace_closest_noalloc: the launch's slot counters, error word
// and stats in the first kNoAllocWordsBytes, then the per-lane stack spill area. Each GPU holds
// its own copy for the life of the process; host code reaches it only through the address that
// noalloc_scratch_lookup returns for the current device.
static __device__ __align__(256) unsigned char scratch[lchip::kNoAllocScratchBytes];

namespace lchip {

// Address of the current device's copy of `scratch`, looked up on the first call for each device
// (with that device current) and kept per device index for later calls.
hipError_t noalloc_scratch_lookup(void **device_ptr) {
    static std::mutex mu;
    static std::map<int, void *> by_device;
    *device_ptr = nullptr;
    int index = 0;
    hipError_t e = hipGetDevice(&index);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lk(mu);
    auto it = by_device.find(index);
    if (it != by_device.end()) {
        *device_ptr = it->second;
        return hipSuccess;
    }
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    by_device.emplace(index, p);
    *device_ptr = p;
    return hipSuccess;
}

// Template parameters: ANY (trace_any), TWO (TLAS + BLAS; otherwise one instance's BLAS),
// COUNT (count node visits / triangle tests), BLOCK threads, SLDS stack entries in LDS.
// With the 8-entry LDS stack the single-level forms fit 6 (<= 80 VGPRs) and the two-level forms 5
// (<= 96 VGPRs) waves per SIMD; the hint keeps the register allocator there (deeper LDS stacks are
// limited by LDS first). None spills but the two-level closest-hit form: 7 VGPRs, and 40 B of scratch
// per lane in all, 8 of them of the eight-lane body.
template<bool ANY, bool TWO, bool COUNT, int BLOCK, int SLDS>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(SLDS == 8 ? (TWO ? 5 : 6) : 1)))
void k_trace(const TraceParams P) {
    __shared__ trav::WaveShared<ANY, BLOCK, SLDS> shared;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t count = P.count_ptr ? min(*P.count_ptr, P.count) : P.count;
    if constexpr (BLOCK == 64 && !COUNT) {
        // A queue counted on the device that turns out short: eight lanes per ray, in as many waves as
        // trace_grid would take and a second round or part of one, spread over the XCDs (the last depths of
        // a 1080p wave of one sample, whose launches are sized for its first: closest 160 -> 65 us, any 140
        // -> 32). The limits on 256 CUs, measured at them, eight lanes per ray / one (which the waves claim):
        // any hit, one level, 98,304 rays: 171 / 263 us (soup of 1M), 210 / 346 (8M), 69 / 201 (sphere of
        // 82k); two levels, 81,920: 206 / 324 (two overlapping soups), 154 / 302 (1,024 instances), 54 / 141
        // (room). Closest hit, one level, 61,440: 238 / 286, 254 / 335, 69 / 207; two levels, 51,200: 222 / 356
        // (1,024 instances), 102 / 174 (room), 304 / 353 (two overlapping soups, camera), and the one case
        // that loses, 531 / 480 (the same, incoherent; 280 / 467 at 40,960).
        constexpr uint32_t kRays = ANY ? 16u : 10u; // per resident wave
        const uint32_t blocks = gridDim.x & ~(kFetchSegments - 1u);
        if (P.simds != 0u && count <= kRays * blocks) {
            uint32_t rays = 1u;
            while (rays < 8u && (count + rays - 1u) / rays > min(P.simds, blocks)) rays *= 2u;
            const uint32_t per_xcd = min(blocks, (count + rays - 1u) / rays + kFetchSegments - 1u) / kFetchSegments;
            if (blockIdx.x >= per_xcd * kFetchSegments) return;
            for (uint32_t w = (blockIdx.x % kFetchSegments) * per_xcd + blockIdx.x / kFetchSegments; w * rays < count;
                 w += per_xcd * kFetchSegments)
                trav::trace_octets<ANY, TWO>(P, reinterpret_cast<uint2 (*)[8]>(&shared.stk[0][0]), w, rays, count);
            return;
        }
    }
    trav::WaveWalker<ANY, TWO, COUNT, BLOCK, SLDS> W;
    W.init(P, &shared, tid);

    const uint64_t rounds = W.trace_queue(P, count); // counting form: refill rounds of this wave
    if (COUNT) {
        // stats: node visits, triangle tests, live lane-iterations, wave iterations, refill rounds
        uint64_t v[5] = {W.n_nodes, W.n_tris, W.n_live, W.n_wave, rounds};
        for (int k = 0; k < 5; k++) {
            for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o, 64);
            if (lane == 0) atomicAdd(reinterpret_cast<unsigned long long *>(P.stats) + k, (unsigned long long)v[k]);
        }
    }
}

// Eight lanes per ray, P.lanes rays per wave (trace_grid); every ray of the launch has its lanes.
template<bool ANY, bool TWO>
__global__ __launch_bounds__(64) void k_trace_oct(const TraceParams P) {
    __shared__ uint2 stk[trav::kOctStack][8];
    const uint32_t count = P.count_ptr ? min(*P.count_ptr, P.count) : P.count;
    // waves XCD by XCD, as in WaveWalker::trace_queue
    const uint32_t w = (blockIdx.x % kFetchSegments) * (gridDim.x / kFetchSegments) + blockIdx.x / kFetchSegments;
    trav::trace_octets<ANY, TWO>(P, stk, w, P.lanes, count);
}

__global__ void k_zero_counter(uint32_t *c) {
    if (threadIdx.x < kFetchSegments) c[threadIdx.x * kCounterStride] = 0u;
}

namespace {

template<bool ANY, bool TWO, bool COUNT, int BLOCK, int SLDS>
hipError_t launch_one(const TraceParams &P, hipStream_t stream, int grid) {
    hipLaunchKernelGGL((k_trace<ANY, TWO, COUNT, BLOCK, SLDS>), dim3(grid), dim3(BLOCK), 0, stream, P);
    return hipGetLastError();
}

template<bool ANY, bool TWO, bool COUNT>
hipError_t launch_cfg(const TraceParams &P, hipStream_t stream, int grid, int block, int slds) {
#define LC_TRACE_CFG(B, S) \
    if (block == B && slds == S) return launch_one<ANY, TWO, COUNT, B, S>(P, stream, grid);
    LC_TRACE_CFG(64, 8) LC_TRACE_CFG(64, 16) LC_TRACE_CFG(64, 24)
    LC_TRACE_CFG(128, 8) LC_TRACE_CFG(128, 16) LC_TRACE_CFG(128, 24)
    LC_TRACE_CFG(256, 8) LC_TRACE_CFG(256, 16) LC_TRACE_CFG(256, 24)
#undef LC_TRACE_CFG
    return hipErrorInvalidValue;
}

template<bool ANY, bool TWO, bool COUNT, int BLOCK, int SLDS>
int occupancy_one() {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, (const void *)k_trace<ANY, TWO, COUNT, BLOCK, SLDS>, BLOCK, 0) != hipSuccess)
        return 1;
    return nb > 0 ? nb : 1;
}

template<bool ANY, bool TWO, bool COUNT>
int occupancy_cfg(int block, int slds) {
#define LC_OCC_CFG(B, S) \
    if (block == B && slds == S) return occupancy_one<ANY, TWO, COUNT, B, S>();
    LC_OCC_CFG(64, 8) LC_OCC_CFG(64, 16) LC_OCC_CFG(64, 24)
    LC_OCC_CFG(128, 8) LC_OCC_CFG(128, 16) LC_OCC_CFG(128, 24)
    LC_OCC_CFG(256, 8) LC_OCC_CFG(256, 16) LC_OCC_CFG(256, 24)
#undef LC_OCC_CFG
    return 1;
}

} // namespace

bool trace_config_supported(int block, int slds) {
    return (block == 64 || block == 128 || block == 256) && (slds == 8 || slds == 16 || slds == 24);
}

int trace_blocks_per_cu(bool any, bool two, bool count, int block, int slds) {
    if (any) {
        if (two) return count ? occupancy_cfg<true, true, true>(block, slds) : occupancy_cfg<true, true, false>(block, slds);
        return count ? occupancy_cfg<true, false, true>(block, slds) : occupancy_cfg<true, false, false>(block, slds);
    }
    if (two) return count ? occupancy_cfg<false, true, true>(block, slds) : occupancy_cfg<false, true, false>(block, slds);
    return count ? occupancy_cfg<false, false, true>(block, slds) : occupancy_cfg<false, false, false>(block, slds);
}

// A launch whose rays all fit the lanes that can be resident hands them out once, without slot
// counters (and without the launch that clears them).
//  - Eight lanes per ray (k_trace_oct) while kOctWaves waves per SIMD hold every ray: 65,536 rays on
//    256 CUs. Measured, one ray per lane against eight lanes per ray, incoherent closest hits: soup of
//    1M triangles, 1,024 rays 108 -> 79 us, 16,384 160 -> 109, 49,152 190 -> 141, 65,536 196 -> 185,
//    98,304 188 -> 214; sphere of 82k, 16,384 83 -> 43, 65,536 81 -> 55; 1,024 instances, 65,536
//    263 -> 187; any hit, soup, 65,536 147 -> 109. Two overlapping soups lose above 45,000 rays
//    (49,152 379 -> 401, 65,536 445 -> 452; their any hits 219 -> 165), at no more than the kernel before
//    (548). The eight lanes do the node decode eight times, so the form loses once the SIMDs have enough
//    waves to be bound by VALU issue.
//  - Otherwise one ray per lane; when that leaves SIMDs without a wave, waves take fewer rays (down
//    to kMinLanes: nearest-commit queries, and traces that count their work): a wave lasts as long
//    as its slowest ray plus the triangle steps of the others, one step after another, each a
//    memory latency.
TraceGrid trace_grid(uint64_t count, int block, int blocks_per_cu, int cu_count, bool octets) {
    constexpr uint32_t kMinLanes = 4, kOctWaves = 8;
    const uint64_t cus = (uint64_t)std::max(1, cu_count);
    const uint64_t most = (uint64_t)std::max(1, blocks_per_cu) * cus;
    const uint64_t waves_per_block = (uint64_t)(block / 64);
    if (count > most / kFetchSegments * kFetchSegments * (uint64_t)block) return {(int)most, 0u, false};
    const uint64_t simds = 4u * cus;
    if (octets && count <= simds * kOctWaves * 8u) {
        uint32_t rays = 1; // per wave
        while (rays < 8u && (count + rays - 1) / rays > simds) rays *= 2u;
        return {(int)(((count + rays - 1) / rays + kFetchSegments - 1) / kFetchSegments * kFetchSegments), rays, true};
    }
    uint32_t lanes = kMinLanes;
    while (lanes < 64u && (count + lanes - 1) / lanes > simds) lanes *= 2u;
    uint64_t grid = ((count + lanes - 1) / lanes + waves_per_block - 1) / waves_per_block;
    grid = (grid + kFetchSegments - 1) / kFetchSegments * kFetchSegments; // k_trace counts waves XCD by XCD
    return {(int)grid, lanes, false};
}

hipError_t trace_launch(const TraceParams &P, hipStream_t stream, bool any, bool two, bool count, int grid, int block,
                        int slds) {
    if (P.octets != 0u && !count) {
        const auto k = any ? (two ? k_trace_oct<true, true> : k_trace_oct<true, false>)
                           : (two ? k_trace_oct<false, true> : k_trace_oct<false, false>);
        hipLaunchKernelGGL(k, dim3(grid), dim3(64), 0, stream, P);
        return hipGetLastError();
    }
    if (P.lanes == 0u)
        hipLaunchKernelGGL(k_zero_counter, dim3(1), dim3(64), 0, stream, P.ray_counter);
    if (any) {
        if (two) return count ? launch_cfg<true, true, true>(P, stream, grid, block, slds) : launch_cfg<true, true, false>(P, stream, grid, block, slds);
        return count ? launch_cfg<true, false, true>(P, stream, grid, block, slds) : launch_cfg<true, false, false>(P, stream, grid, block, slds);
    }
    if (two) return count ? launch_cfg<false, true, true>(P, stream, grid, block, slds) : launch_cfg<false, true, false>(P, stream, grid, block, slds);
    return count ? launch_cfg<false, false, true>(P, stream, grid, block, slds) : launch_cfg<false, false, false>(P, stream, grid, block, slds);
}

} // namespace lchip
