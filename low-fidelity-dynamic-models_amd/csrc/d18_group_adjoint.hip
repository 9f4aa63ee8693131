// Differentiation form of the 18-DOF solver on lane groups: the forward and the reverse sweep of
// d18_adjoint.hip with each vehicle on two or four lanes (d18_group_adjoint.h), same buffers, same bits.
#include <hip/hip_runtime.h>

#include "d18_group_adjoint.h"
#include "integrate.h"

namespace lfdm {

using namespace dev;

namespace {

constexpr int kThreads = 64;

// This lane's slot and place, and the maps of its wavefront's set in LDS; false past the fleet's end.
template <int G>
__device__ __forceinline__ bool group_lane(const AdjLaunch& L, MapXY* tab, int& slot, int& q, const PSet*& P) {
    slot = (int)((blockIdx.x * blockDim.x + threadIdx.x) / G);
    q = (int)(threadIdx.x % G);
    const int wave = uniform(slot >> 6);
    if (wave * kWave >= L.S) return false;
    P = &pset_at(L.sets, uniform(L.wave_set[wave]));
    kern::stage_maps(*P, tab, (int)(threadIdx.x % kWave));
    return true;
}

template <int G, int W>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(W, W))) void adj_forward_g(AdjLaunch L) {
    __shared__ MapXY tab[kGroupMapEntries];
    int slot, q;
    const PSet* P;
    if (!group_lane<G>(L, tab, slot, q, P)) return;
    adj_forward_group<G, W == 1>(L, slot, q, *P, tab);
}

// The constants and their adjoints lie in LDS (ReverseStore): in registers they would take 88 of a lane's
// (468 instead of 368 on four lanes).
template <int G>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void adj_reverse_g(AdjLaunch L) {
    __shared__ MapXY tab[kGroupMapEntries];
    __shared__ ReverseStore<G, kThreads> store;
    int slot, q;
    const PSet* P;
    if (!group_lane<G>(L, tab, slot, q, P)) return;
    adj_reverse_group<G>(L, slot, q, *P, tab, store.constants(threadIdx.x), store.adjoints(threadIdx.x));
}

template <int G>
unsigned grid(const AdjLaunch& L) {
    return (unsigned)(((long long)L.S * G + kThreads - 1) / kThreads);
}

}  // namespace

hipError_t launch_adj_forward_group(const AdjLaunch& L, KernelChoice c, hipStream_t stream) {
    if (L.S <= 0 || L.nsteps <= 0) return hipSuccess;
    if (c.lanes == 4 && c.waves == 1)
        hipLaunchKernelGGL((adj_forward_g<4, 1>), grid<4>(L), kThreads, 0, stream, L);
    else if (c.lanes == 4)
        hipLaunchKernelGGL((adj_forward_g<4, 2>), grid<4>(L), kThreads, 0, stream, L);
    else
        hipLaunchKernelGGL((adj_forward_g<2, 2>), grid<2>(L), kThreads, 0, stream, L);
    return hipGetLastError();
}

hipError_t launch_adj_reverse_group(const AdjLaunch& L, int lanes, hipStream_t stream) {
    if (L.S <= 0 || L.seg_hi <= L.seg_lo) return hipSuccess;
    if (lanes == 4)
        hipLaunchKernelGGL(adj_reverse_g<4>, grid<4>(L), kThreads, 0, stream, L);
    else
        hipLaunchKernelGGL(adj_reverse_g<2>, grid<2>(L), kThreads, 0, stream, L);
    return hipGetLastError();
}

}  // namespace lfdm
