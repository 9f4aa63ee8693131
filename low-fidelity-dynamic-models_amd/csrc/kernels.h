// Launch records and host-side entry points of the HIP kernels.
//
// Records (one per vehicle; SoA on the device as [field][slot]); the full field lists are in
// integrate.h:
//   11-DOF  2 tires x 15 (TMeasy) / 11 (TMeasyNr) + 12 vehicle fields       = 42 / 34
//   18-DOF  4 tires x 15 / 11 + 15 vehicle fields                           = 75 / 59
//   24-DOF  4 tires x 23 / 19 + 4 struts x 24 + 24 vehicle fields           = 212 / 196
#pragma once
#include <hip/hip_runtime.h>

#include "lfdm_types.h"

namespace lfdm {

// Parameter set i of a launch.  Sets are never written while a kernel runs, so they are read
// through the constant address space: reads at a wave-uniform address then become scalar loads into
// SGPRs instead of vector loads into VGPR pairs (which also lowers the step's VGPR pressure).
__device__ __forceinline__ const PSet& pset_at(const PSet* sets, int i) {
    return *(const PSet*)((const __attribute__((address_space(4))) PSet*)sets + i);
}

// Most waves per SIMD each model's integration kernels are built for (each also exists at every lower
// occupancy; the maximum is the default on fleets of more than one wavefront per SIMD).
constexpr int kMaxWaves11 = 4, kMaxWaves18 = 3, kMaxWaves24 = 2;

// Lanes per vehicle and waves per SIMD of the kernel a fleet of S slots runs on a device of `simds` SIMDs
// (waves 0: the model's most).  A lone wavefront on a SIMD leaves most of its cycles unused, and a
// fleet of few wavefronts leaves SIMDs idle, so such fleets spread each vehicle over a group of lanes
// (csrc/group.h): every lane then has one or two tires instead of four and shares the map lookups and
// angles.  Measured per step (TMeasy fleets, microseconds; one lane / two / four):
//   18-DOF  16,384 vehicles  7.8 / 4.0 / 2.5    32,768  8.1 / 4.2 / 4.1    65,536  8.3 / 6.1 / 7.7
//   24-DOF  16,384 vehicles  9.9 / 5.4 / 3.2    32,768 10.3 / 5.3 / 4.9    65,536 10.3 / 8.3 / 9.8
//   11-DOF  16,384 vehicles  4.9 / 2.4          32,768  5.5 / 2.4          65,536  5.7 / 3.9
// TMeasyNr fleets, whose tires take longer, gain likewise (65,536 vehicles, one / two: 18-DOF 11.7 / 9.5, 24-DOF 13.0 /
// 11.0, 11-DOF 7.3 / 5.4; 16,384, one / four: 18-DOF 11.6 / 3.4, 24-DOF 12.6 / 3.9).
// So: four lanes while they make at most two wavefronts per SIMD, two lanes while they do, and one lane
// beyond (at 131,072 18-DOF vehicles two lanes would take two rounds of 6.1 against 10.8).  The kernels are
// built for the wavefronts per SIMD they make, which keeps the dispatcher from stacking two on one SIMD
// while another is idle.  One-lane fleets of w wavefronts per SIMD, w below the model's most, run the
// kernel built for w for the same reason.  one_lane: launches that have no lane-group kernels (the strict step,
// a caller's own controls functor).
struct KernelChoice {
    int lanes, waves;
};

inline KernelChoice choose_kernel(int dof, long long S, int simds, bool one_lane) {
    const long long wf = S / kWave;
    if (simds <= 0 || wf <= 0) return {1, 0};
    const auto per = [&](int lanes) { return (wf * lanes + simds - 1) / simds; };
    if (!one_lane) {
        if (dof != 11 && per(4) <= 2) return {4, (int)per(4)};
        if (per(2) <= 2) return {2, dof == 11 ? (int)per(2) : 2};
    }
    const int most = dof == 11 ? kMaxWaves11 : dof == 18 ? kMaxWaves18 : kMaxWaves24;
    return {1, per(1) < most ? (int)per(1) : 0};
}

// Lanes per vehicle of the adjoint's reverse sweep (its forward follows choose_kernel).  Its step holds more
// registers than two wavefronts per SIMD have (256 per lane would spill 106 on four lanes, 204 on two: 16,384
// vehicles 13.0 us per step instead of 6.6, 65,536 on two lanes 37 instead of 17.8 on one), so a vehicle gets
// more lanes only while they make one wavefront per SIMD at most.  Per step (us) on one lane / two / four:
//   16,384 vehicles 17.0 / 10.1 / 6.6    32,768 17.0 / 10.6 / -    65,536 17.8 / 21.3 (two rounds)
inline int reverse_lanes(long long S, int simds) {
    const long long wf = S / kWave;
    return wf * 4 <= simds ? 4 : wf * 2 <= simds ? 2 : 1;
}

struct Launch {
    const PSet* sets;       // parameter sets
    const int* wave_set;   // set index of every 64-slot wavefront
    const int* slot_user;  // user vehicle index of every slot, -1 for padding
    double* state;         // [record field][S]
    const double* ovr;     // [kOverrides][S]
    const DrvRow* drv;     // driver-table pool (kCtrlTable)
    const double* knots;   // [ns + 2 np][n_user] (kCtrlKnots)
    const double* steps;   // [nsteps][3][n_user] for this launch (kCtrlSteps)
    const int* out_steps;  // step counts after which an output row is written, ascending
    double* out;           // [n_out][channels][n_user]
    double t0, dt;
    double c_s, c_t, c_b;  // kCtrlConst
    double ds, dp;         // knot spacings (kCtrlKnots)
    int ns, np;
    int nsteps, n_out, S, n_user, mode, nr;
    int steps_shared;      // kCtrlSteps: 1 = steps[nsteps][3] shared by every vehicle
    // per-vehicle horizons (null: every vehicle runs all nsteps): a vehicle stops after
    // horizon[slot] steps counted from step 0 of the solve; step_base steps were done before this
    // launch; wave_hmax[wave] is the largest horizon of the wavefront
    const int* horizon;
    const int* wave_hmax;
    int step_base;
    int waves;  // waves per SIMD of the kernel: 1 up to the model's maximum, or 0 for its default
    int lanes;  // lanes per vehicle: 0 or 1 the one-lane kernels, 2 or 4 the lane-group kernels (not for strict)
    int strict;  // 1: the step with the reference's own quotients and transcendentals (LFDM_ARITH_STRICT)
};

// Integration launches of the 11-, 18- and 24-DOF models (one kernel per tire model and control
// source inside each).
hipError_t launch_d11(const Launch& L, int block, hipStream_t stream);
hipError_t launch_d18(const Launch& L, int block, hipStream_t stream);
hipError_t launch_d24(const Launch& L, int block, hipStream_t stream);
hipError_t launch_d11_group(const Launch& L, int block, hipStream_t stream);
hipError_t launch_d24_group(const Launch& L, int block, hipStream_t stream);
hipError_t launch_d18_group(const Launch& L, int block, hipStream_t stream);

// Differentiation form (18-DOF TMeasy).  Forward: from the record state, nsteps steps with per-step
// controls ctrl[nsteps][3][n_user]; writes xy[nsteps][2][n_user] (position after each step) and
// the carried state every K steps into ckpt[ceil(nsteps/K)][32][S].  Backward, one group of
// segments [seg_lo, seg_hi) at a time, last group first: the recompute launch reruns the group's
// segments from their checkpoints into tape[seg_hi - seg_lo][S / 64][K][38][64] (the carried state and
// tire outputs the step adjoint reads, every step, blocked by wavefront), the reverse launch walks them backwards.  From xy_bar (layout of xy) the
// last group's reverse writes ctrl_bar (layout of ctrl), state_bar[75][n_user] (adjoint of the
// initial record) and param_bar[7][n_user] (m, jz, jx, dfy0Pn, dfy0P2n, torque scale,
// maxBrakeTorque); between groups the running adjoints live in carry[52][S].
constexpr int kAdjCkptRow = 32;  // doubles per vehicle in a checkpoint
constexpr int kAdjTapeRow = 38;  // doubles per vehicle and step in the tape
constexpr int kAdjCarry = 52;    // doubles per vehicle in carry

struct AdjLaunch {
    const PSet* sets;
    const int* wave_set;
    const int* slot_user;
    const double* state;
    const double* ovr;
    const double* ctrl;
    double* xy;
    const double* xy_bar;
    double* ctrl_bar;
    double* state_bar;
    double* param_bar;
    double* ckpt;
    double* tape;
    double* carry;
    double dt;
    int nsteps, K, S, n_user;
    int seg_lo, seg_hi;  // backward: the group of this launch
    int fwd_tape_lo;     // forward: segments from this one on also go to the tape (block 0 onwards)
    double* jac;         // step Jacobian: [kJacRows][kJacCols][n_user]
};

// Step Jacobian (lfdm_step_jacobian): rows are the stepped packed states, columns the packed states
// then steering, throttle and braking, both in the reference's packY order of a vehicle with a torque
// converter (xe ye per tire, omega x 4, crankOmega, x y u v psi wz phi wx).
constexpr int kJacRows = 21;
constexpr int kJacCols = kJacRows + 3;

// The forward pass: one lane per vehicle on fleets of more than one wavefront per SIMD, else on lane groups.
hipError_t launch_adj_forward(const AdjLaunch& L, hipStream_t stream);
hipError_t launch_adj_forward_group(const AdjLaunch& L, KernelChoice c, hipStream_t stream);
hipError_t launch_adj_reverse_group(const AdjLaunch& L, int lanes, hipStream_t stream);
hipError_t launch_adj_recompute(const AdjLaunch& L, hipStream_t stream);
hipError_t launch_adj_reverse(const AdjLaunch& L, hipStream_t stream);
// Every vehicle's step Jacobian at its current record under the per-vehicle controls ctrl[3][n_user].
hipError_t launch_step_jacobian(const AdjLaunch& L, hipStream_t stream);

// Records `msg` as the calling thread's lfdm_last_error() text and returns `code`.
int set_last_error(int code, const char* msg);

// Gathers full records of `n` slots from SoA state into out[n][rec].
hipError_t launch_gather(const double* state, int S, int rec, const int* slots, int n, double* out,
                         hipStream_t stream);
// Scatters field-major rows src[F][n] (vehicle v in column v) into dst[F][S] at user_slot[v].
hipError_t launch_scatter_fields(double* dst, int S, int F, const int* user_slot, int n, const double* src,
                                 hipStream_t stream);
// Scatters records in[n][rec] into the SoA state at `slots`.
hipError_t launch_scatter(double* state, int S, int rec, const int* slots, int n, const double* in,
                          hipStream_t stream);

}  // namespace lfdm
