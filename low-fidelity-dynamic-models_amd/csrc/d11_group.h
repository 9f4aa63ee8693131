// The 11-DOF step on two lanes (lane 0 the front tire, lane 1 the rear), fast arithmetic form.  Same
// operations in the same order as step11 for every value, so the same bits.
#pragma once
#include "d11_device.h"
#include "group.h"

namespace lfdm {
namespace dev {

// Carried state of one lane: its own tire and the whole chassis.
struct S11g {
    int q;  // this lane's place in the group
    double xe, ye, xedot, yedot, omega;
    double x, y, u, v, psi, wz, udot, crank;
    int gear;
    Walks<2> maps;
    GearRow row;
};

// Per-vehicle constants, and those of this lane's tire.
struct K11g {
    K11 c;
    bool front, walks;
    double Z, Z4n, arm;  // the load transfer carries the axle's sign (negation is exact)
};

LFDM_HD void k11g_init(const PSet& P, const K11& c, int q, K11g& k) {
    k.c = c;
    k.front = q == 0;
    k.walks = group_walks(P);
    k.Z = k.front ? c.Z1 : c.Z3;
    k.Z4n = k.front ? -c.Z4n : c.Z4n;
    k.arm = k.front ? P.a : -P.b;
}

// What the last step's record holds of this lane's tire (the chassis part on both lanes).
struct X11g {
    double dOmega, xt, rStat, fx, fy, fz, vsx, vsy, My, engTor;
    double vdot, wzdot, dcrank;
};

// x, y and psi from the new velocities at the yaw angle's sine and cosine, as position11 does.
LFDM_HD void move11g(S11g& s, double sp, double cp, double dt) {
    s.x = s.x + (s.u * cp - s.v * sp) * dt;
    s.y = s.y + (s.u * sp + s.v * cp) * dt;
    s.psi = s.psi + s.wz * dt;
}

// step11 without its closing position update; `lag`: the previous step's position update comes first
// (its sine and cosine of the yaw angle from lane 1 while lane 0 takes the steering angle's).
template <bool NR, bool FULL, class PS>
LFDM_HD void step11g(const PS& P, const Derived& u, const K11g& k, S11g& s, double steering, double throttle,
                     double braking, double dt, bool lag, X11g* x) {
    const TireP& t = P.tire;
    const double delta = P.nonLinearSteer ? map_y<false>(full_set(P).steer, steering) : steering * P.maxSteer;
    double sa, ca;
    sincos_fast((s.q & 1) ? s.psi : delta, sa, ca);
    const double sd = group_value<2, 0>(sa), cd = group_value<2, 0>(ca);
    if (lag) move11g(s, group_value<2, 1>(sa), group_value<2, 1>(ca), dt);
    // computeTireLoads
    const double Z2 = fdiv(k.Z4n * (s.udot - s.wz * s.v), k.c.two_ab);
    double fz = k.Z + Z2;
    fz = fz > 0. ? fz : 0.;
    // wheel speeds as the powertrain will read them: a tire off the ground resets its own
    const double om = fz <= 0 ? 0 : s.omega;
    const double omf = group_value<2, 0>(om), omr = group_value<2, 1>(om);
    // the powertrain's torque: nothing in it depends on this step's tire forces
    double shaft, dcrank;
    powertrain_group<2>(P, u, k.c.tqs, throttle, s.u, 0.5 * (omf + omr), s.q, k.walks, s.maps, s.row, s.crank, s.gear,
                        shaft, dcrank);
    double engf, engr;
    if (P.driveType) {
        diff_split<false>(shaft, omr, omf, engr, engf);
    } else if (P.whichWheels) {
        engr = shaft;
        engf = 0;
    } else {
        engr = 0;
        engf = shaft;
    }
    const double eng = k.front ? engf : engr;
    // vehToTireTransform
    const double vsy = s.v + s.wz * k.arm;
    const double vf = s.u * cd + vsy * sd;
    const double vsx = k.front ? vf : s.u;
    // computeTireRHS
    const double tand = fdiv(sd, cd);
    const double d = k.front ? tand : u.tan_delta_rear;
    double fx, fy, My, xt, rStat;
    if (fz <= 0) {
        if (!NR) { s.xe = 0; s.ye = 0; }
        s.omega = 0; xt = 0; rStat = t.r0; fx = 0; fy = 0; My = 0;
    } else {
        xt = fz * u.inv_kt;
        rStat = t.r0 - xt;
        if (!NR)
            tmeasy_core<false>(t, u, k.c.qy1, k.c.qy2, 0.0, d, fz, rStat, vsx, vsy, s.xe, s.ye, s.omega, s.xedot,
                               s.yedot, fx, fy, My);
        else
            tmeasy_nr_core<false>(t, u, k.c.qy1, k.c.qy2, 0.0, d, fz, rStat, vsx, vsy, s.omega, fx, fy, My);
    }
    const double bt = k.c.maxBrake * braking;
    const double dOm = u.inv_jw * (eng + My - sgn(s.omega) * bt - fx * rStat);
    // tireToVehTransform (front tire only)
    {
        const double gx = fx * cd - fy * sd;
        const double gy = fx * sd + fy * cd;
        fx = k.front ? gx : fx;
        fy = k.front ? gy : fy;
    }
    const double fxf = group_value<2, 0>(fx), fxr = group_value<2, 1>(fx);
    const double fyf = group_value<2, 0>(fy), fyr = group_value<2, 1>(fy);
    // computeVehRHS
    const double vdot = -s.u * s.wz + fdiv(fyf + fyr, k.c.mt);
    const double udot = s.v * s.wz + fdiv(fxf + fxr, k.c.mt);
    const double wzdot = fdiv(P.a * fyf - P.b * fyr, k.c.jz);
    if (!NR) {
        s.xe = s.xe + s.xedot * dt;
        s.ye = s.ye + s.yedot * dt;
    }
    s.omega = s.omega + dOm * dt;
    if (P.tcbool) s.crank = s.crank + dcrank * dt;
    s.u = s.u + udot * dt;
    s.v = s.v + vdot * dt;
    s.wz = s.wz + wzdot * dt;
    s.udot = udot;
    if (FULL) {
        x->dOmega = dOm; x->xt = xt; x->rStat = rStat; x->fx = fx; x->fy = fy;
        x->fz = fz; x->vsx = vsx; x->vsy = vsy; x->My = My; x->engTor = eng;
        x->vdot = vdot;
        x->wzdot = wzdot;
        x->dcrank = dcrank;
    }
}

}  // namespace dev
}  // namespace lfdm
