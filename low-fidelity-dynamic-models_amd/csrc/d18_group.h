// The 18-DOF step on a group of G lanes (2: an axle per lane, 4: a tire per lane), fast arithmetic
// form.  Same operations in the same order as step18 for every value, so the same bits.
#pragma once
#include "d18_device.h"
#include "group.h"

namespace lfdm {
namespace dev {

// Carried state of one lane: its own N = 4 / G tires (first tire N q) and the whole chassis.
template <int G>
struct S18g {
    static constexpr int N = 4 / G;
    int q;  // this lane's place in the group
    double xe[N], ye[N], xedot[N], yedot[N], omega[N];
    double x, y, u, v, psi, wz, phi, wx, udot, vdot, crank;
    int gear;
    Walks<G> maps;
    GearRow row;
};

// Constants of this lane's axle or tire (beside the vehicle's K18): with a tire per lane the load
// transfers and the half track carry its side's sign (negation is exact), so that one expression
// serves all four.
template <int G>
struct K18g {
    bool front, walks;
    double Z1, Z2c, kro, bro, inv_c, inv_two_ab, track, arm;
};

template <int G>
LFDM_HD void k18g_init(const PSet& P, const K18& c, int q, K18g<G>& k) {
    k.front = G == 4 ? q < 2 : q == 0;
    k.walks = group_walks(P);
    const double side = G == 4 && (q & 1) == 0 ? -1.0 : 1.0;  // a left tire's lane: minus
    k.Z1 = k.front ? c.Z1f : c.Z1r;
    k.Z2c = side * (k.front ? c.Z2fc : c.Z2rc);
    k.kro = side * (k.front ? P.krof : P.kror);
    k.bro = side * (k.front ? P.brof : P.bror);
    k.inv_c = k.front ? P.d.inv_cf : P.d.inv_cr;
    k.inv_two_ab = k.front ? -P.d.inv_two_ab : P.d.inv_two_ab;
    k.track = side * (k.front ? P.cf : P.cr);
    k.arm = k.front ? P.a : -P.b;
}

// What the last step's record holds of this lane's tires (the chassis part on every lane).
template <int G>
struct X18g {
    static constexpr int N = 4 / G;
    double dOmega[N], xt[N], rStat[N], fx[N], fy[N], fz[N], vsx[N], vsy[N], My[N], engTor[N];
    double wxdot, wzdot, dcrank;
};

// x, y and psi from the new velocities at the yaw angle's sine and cosine, as position18 does.
template <int G>
LFDM_HD void move18g(S18g<G>& s, double sp, double cp, double dt) {
    s.x = s.x + (s.u * cp - s.v * sp) * dt;
    s.y = s.y + (s.u * sp + s.v * cp) * dt;
    s.psi = s.psi + s.wz * dt;
}

// The step's steering angle, with the previous step's position update (`lag`): one lane takes the sine and
// cosine of the steering angle while another takes the yaw angle's.
template <int G, class PS>
LFDM_HD void angles18g(const PS& P, S18g<G>& s, double steering, double dt, bool lag, double& sd, double& cd) {
    const double delta = P.nonLinearSteer ? map_y<false>(full_set(P).steer, steering) : steering * P.maxSteer;
    double sa, ca;
    sincos_fast((s.q & 1) ? s.psi : delta, sa, ca);
    sd = group_value<G, 0>(sa);
    cd = group_value<G, 0>(ca);
    if (lag) move18g<G>(s, group_value<G, 1>(sa), group_value<G, 1>(ca), dt);
}

// A lane's tire right-hand-side outputs of one step (before the front forces are rotated), for the tape.
template <int G>
struct TireOut18g {
    static constexpr int N = 4 / G;
    double fx[N], fy[N], My[N], rStat[N];
};

// This lane's wheel loads, before the clamp at zero.
template <int G>
LFDM_HD void loads18g(const K18& c, const K18g<G>& k, double lat, double phi, double wx, double udot, double wz, double v,
                      double* fz) {
    const double Z2 = k.Z2c * lat;
    const double Z3 = (k.kro * phi + k.bro * wx) * k.inv_c;
    const double Z4 = (c.Z4n * (udot - wz * v)) * k.inv_two_ab;
    if constexpr (G == 4) {
        fz[0] = k.Z1 + Z2 + Z3 + Z4;
    } else {
        fz[0] = k.Z1 - Z2 - Z3 + Z4;
        fz[1] = k.Z1 + Z2 + Z3 + Z4;
    }
}

// This lane's contact-patch velocities; returns the lateral one, the longitudinal ones in vsx.
template <int G>
LFDM_HD double patch18g(const K18g<G>& k, double u, double v, double wz, double sd, double cd, double* vsx) {
    const double vsy = v + wz * k.arm;
    const double hw = (wz * k.track) / 2.;
#pragma unroll
    for (int j = 0; j < 4 / G; ++j) {
        const double vx = G == 4 || j == 1 ? u + hw : u - hw;
        const double vf = vx * cd + vsy * sd;
        vsx[j] = k.front ? vf : vx;
    }
    return vsy;
}

// step18 without its closing position update, after angles18g.
template <bool NR, bool FULL, int G, bool CAPTURE = false, class PS>
LFDM_HD void step18g(const PS& P, const Derived& u, const K18& c, const K18g<G>& k, S18g<G>& s, double sd, double cd,
                     double throttle, double braking, double dt, X18g<G>* x, TireOut18g<G>* to = nullptr) {
    constexpr int N = 4 / G;
    const TireP& t = P.tire;
    // computeTireLoads
    double fz[N];
    loads18g<G>(c, k, s.vdot + s.wz * s.u, s.phi, s.wx, s.udot, s.wz, s.v, fz);
#pragma unroll
    for (int j = 0; j < N; ++j) fz[j] = fz[j] > 0. ? fz[j] : 0.;
    // wheel speeds as the powertrain will read them: a tire off the ground resets its own (tire_tmeasy)
    double om[N], om4[4];
#pragma unroll
    for (int j = 0; j < N; ++j) om[j] = fz[j] <= 0 ? 0 : s.omega[j];
    group_tires<G>(om, om4);
    // the powertrain's torque: nothing in it depends on this step's tire forces, so it comes first and
    // its dependent chain overlaps the tire's
    double shaft, dcrank;
    powertrain_group<G>(P, u, c.tqs, throttle, s.u, 0.25 * (om4[0] + om4[1] + om4[2] + om4[3]), s.q, k.walks, s.maps,
                        s.row, s.crank, s.gear, shaft, dcrank);
    double tf, tr;
    axle_torques(P, shaft, tf, tr);
    double eng[N];
    {
        double l, r;
        diff_split<false>(k.front ? tf : tr, k.front ? om4[0] : om4[2], k.front ? om4[1] : om4[3], l, r);
        if constexpr (G == 4) {
            eng[0] = (s.q & 1) ? r : l;
        } else {
            eng[0] = l;
            eng[1] = r;
        }
    }
    // vehToTireTransform
    double vsx[N];
    const double vsy = patch18g<G>(k, s.u, s.v, s.wz, sd, cd, vsx);
    // computeTireRHS
    const double tand = fdiv(sd, cd);
    const double d = k.front ? tand : u.tan_delta_rear;
    double fx[N], fy[N], My[N], xt[N], rStat[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        if (!NR)
            tire_tmeasy<false>(t, u, c, 0.0, d, fz[j], vsx[j], vsy, s.xe[j], s.ye[j], s.xedot[j], s.yedot[j],
                               s.omega[j], fx[j], fy[j], My[j], xt[j], rStat[j]);
        else
            tire_tmeasy_nr<false>(t, u, c, 0.0, d, fz[j], vsx[j], vsy, s.omega[j], fx[j], fy[j], My[j], xt[j],
                                  rStat[j]);
    }
    if (CAPTURE) {
#pragma unroll
        for (int j = 0; j < N; ++j) {
            to->fx[j] = fx[j]; to->fy[j] = fy[j]; to->My[j] = My[j]; to->rStat[j] = rStat[j];
        }
    }
    const double bt = c.maxBrake * braking;
    double dOm[N];
#pragma unroll
    for (int j = 0; j < N; ++j) dOm[j] = u.inv_jw * (eng[j] + My[j] - sgn(s.omega[j]) * bt - fx[j] * rStat[j]);
    // tireToVehTransform (front tires only)
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const double gx = fx[j] * cd - fy[j] * sd;
        const double gy = fx[j] * sd + fy[j] * cd;
        fx[j] = k.front ? gx : fx[j];
        fy[j] = k.front ? gy : fy[j];
    }
    double fx4[4], fy4[4];
    group_tires<G>(fx, fx4);
    group_tires<G>(fy, fy4);
    double udot, vdot, wxdot, wzdot;
    chassis18<false>(P, u, c, s.u, s.v, s.wz, s.wx, s.phi, fx4, fy4, udot, vdot, wxdot, wzdot);
#pragma unroll
    for (int j = 0; j < N; ++j) {
        if (!NR) {
            s.xe[j] = s.xe[j] + s.xedot[j] * dt;
            s.ye[j] = s.ye[j] + s.yedot[j] * dt;
        }
        s.omega[j] = s.omega[j] + dOm[j] * dt;
    }
    if (P.tcbool) s.crank = s.crank + dcrank * dt;
    s.u = s.u + udot * dt;
    s.v = s.v + vdot * dt;
    s.wx = s.wx + wxdot * dt;
    s.wz = s.wz + wzdot * dt;
    s.phi = s.phi + s.wx * dt;
    s.udot = udot;
    s.vdot = vdot;
    if (FULL) {
#pragma unroll
        for (int j = 0; j < N; ++j) {
            x->dOmega[j] = dOm[j]; x->xt[j] = xt[j]; x->rStat[j] = rStat[j]; x->fx[j] = fx[j]; x->fy[j] = fy[j];
            x->fz[j] = fz[j]; x->vsx[j] = vsx[j]; x->vsy[j] = vsy; x->My[j] = My[j]; x->engTor[j] = eng[j];
        }
        x->wxdot = wxdot;
        x->wzdot = wzdot;
        x->dcrank = dcrank;
    }
}

}  // namespace dev
}  // namespace lfdm
