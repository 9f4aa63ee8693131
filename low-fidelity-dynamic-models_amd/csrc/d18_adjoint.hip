// Differentiation form of the 18-DOF solver.
//  - adj_forward: integrates with per-step controls, records the (x, y) trajectory and stores the
//    carried state every K steps.
//  - adj_recompute: one lane per (segment of a group, vehicle slot); reruns the segment from its
//    checkpoint into the tape.  Segments are independent, so a group of G segments gives G times
//    the wavefronts of the fleet and the recompute runs at full occupancy even for fleets that fill
//    only one wavefront per SIMD.  The tape is blocked by wavefront (one contiguous 19 KB run per
//    wavefront and step) and the per-vehicle constants sit in LDS.
//  - step_jacobian: one lane per (row, slot); the step's Jacobian at the current record, one step adjoint
//    sweep per row.
//  - adj_reverse: one lane per slot; walks the group's segments backwards through the step adjoint
//    of d18_adjoint.h.  The step adjoint needs the whole register file of a SIMD, so the per-vehicle
//    constants and their adjoints live in LDS (23 + 21 doubles per lane; both structs have an odd
//    number of doubles, so a wavefront's 64-bit LDS accesses at that stride hit distinct banks).
//
// One vehicle per lane as in the integration kernels; every lane of a wave runs the same step
// counts, so the segment loops are wave-uniform.
#include <hip/hip_runtime.h>

#include "d18_adjoint_lanes.h"

namespace lfdm {

using namespace dev;

namespace {

constexpr int kThreads = 256;

// Waves per SIMD of the segment recompute (three: its 164 VGPRs fit without spills, and the group's
// (segment, vehicle) lanes fill them).
#ifndef LFDM_ADJ_RECOMPUTE_WAVES
#define LFDM_ADJ_RECOMPUTE_WAVES 3
#endif

static_assert(sizeof(K18) % 16 == 8 && sizeof(K18b) % 16 == 8, "odd number of doubles per lane in LDS");

// Two waves per SIMD: fleets of no more than one run on lane groups (choose_kernel).
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void adj_forward(AdjLaunch L) {
    const int slot = blockIdx.x * blockDim.x + threadIdx.x;
    const int wave = uniform(slot >> 6);
    if (wave * kWave >= L.S) return;
    adj_forward_lane(L, slot, pset_at(L.sets, uniform(L.wave_set[wave])));
}

__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(LFDM_ADJ_RECOMPUTE_WAVES,
                                                                            LFDM_ADJ_RECOMPUTE_WAVES))) void
adj_recompute(AdjLaunch L) {
    const size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    // S is a multiple of the wavefront size, so q and the slot's wave are wave-uniform
    const int q = uniform((int)(id / (size_t)L.S));
    const int slot = (int)(id - (size_t)q * L.S);
    if (q >= L.seg_hi - L.seg_lo) return;
    __shared__ K18 ks[kThreads];
    adj_recompute_lane(L, q, slot, pset_at(L.sets, uniform(L.wave_set[slot >> 6])), ks[threadIdx.x]);
}

__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void adj_reverse(AdjLaunch L) {
    __shared__ K18 ks[kThreads];
    __shared__ K18b kbs[kThreads];
    const int slot = blockIdx.x * blockDim.x + threadIdx.x;
    const int wave = uniform(slot >> 6);
    if (wave * kWave >= L.S) return;
    adj_reverse_lane(L, slot, pset_at(L.sets, uniform(L.wave_set[wave])), ks[threadIdx.x], kbs[threadIdx.x]);
}

// One wavefront per (row, 64 slots), the rows with most work first, each row through the parts of the step it
// reaches.  With a vehicle's 21 rows on one lane the kernel took the latency of 21 sweeps at any size and ran a
// fleet of 1,563 wavefronts in two rounds: 64 vehicles 580 -> 27 us, 100,003 vehicles 2,479 -> 428 us (0.94 TB/s
// of Jacobian).  One wave per SIMD (330 VGPRs): two, with 102 spilled, measure the same.
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(1, 1))) void step_jacobian(AdjLaunch L) {
    const int slot = blockIdx.x * kWave + threadIdx.x;
    jac_row(L, kJacRows - 1 - (int)blockIdx.y, slot, pset_at(L.sets, uniform(L.wave_set[blockIdx.x])));
}

}  // namespace

hipError_t launch_step_jacobian(const AdjLaunch& L, hipStream_t stream) {
    if (L.S <= 0) return hipSuccess;
    hipLaunchKernelGGL(step_jacobian, dim3(L.S / kWave, kJacRows), kWave, 0, stream, L);
    return hipGetLastError();
}

hipError_t launch_adj_forward(const AdjLaunch& L, hipStream_t stream) {
    if (L.S <= 0 || L.nsteps <= 0) return hipSuccess;
    hipLaunchKernelGGL(adj_forward, (L.S + kThreads - 1) / kThreads, kThreads, 0, stream, L);
    return hipGetLastError();
}

hipError_t launch_adj_recompute(const AdjLaunch& L, hipStream_t stream) {
    const size_t lanes = (size_t)(L.seg_hi - L.seg_lo) * (size_t)L.S;
    if (L.S <= 0 || lanes == 0) return hipSuccess;
    hipLaunchKernelGGL(adj_recompute, (unsigned)((lanes + kThreads - 1) / kThreads), kThreads, 0, stream, L);
    return hipGetLastError();
}

hipError_t launch_adj_reverse(const AdjLaunch& L, hipStream_t stream) {
    if (L.S <= 0 || L.seg_hi <= L.seg_lo) return hipSuccess;
    hipLaunchKernelGGL(adj_reverse, (L.S + kThreads - 1) / kThreads, kThreads, 0, stream, L);
    return hipGetLastError();
}

}  // namespace lfdm
