// The 24-DOF step on a group of G lanes (2: an axle's corners per lane, 4: a corner, tire and strut, per
// lane), fast arithmetic form.  Same operations in the same order as step24 for every value, so the same
// bits.
#pragma once
#include "d24_device.h"
#include "group.h"

namespace lfdm {
namespace dev {

// Carried state of one lane: its own N = 4 / G corners (first corner N q) and the whole chassis.
template <int G>
struct S24g {
    static constexpr int N = 4 / G;
    int q;  // this lane's place in the group
    double xe[N], ye[N], xedot[N], yedot[N], xt[N], omega[N], rStat[N];
    double xs[N], wu[N], dxs[N], fzd[N];
    double x, y, u, v, w, psi, phi, theta, wx, wy, wz;
    double udot, vdot, wdot, wxdot, wydot, wzdot, crank;
    int gear;
    Walks<G> maps;
    GearRow row;
};

// Per-vehicle constants and those of this lane's axle and corners (the half track carries a corner's
// side, the axle distance its end: negation is exact).
template <int G>
struct K24g {
    static constexpr int N = 4 / G;
    double xsi[N], lsi[N], vsz[N];
    double tqs, maxBrake, qy1, qy2, inv_m, inv_jx, inv_jy, inv_jz, half_cf, half_cr;
    double mu, mu_g, inv_mu, hrc, inv_c, track, arm;
    bool front, walks;
};

template <int G>
LFDM_HD void k24g_init(const PSet& P, const K24& c, int q, K24g<G>& k) {
    k.tqs = c.tqs; k.maxBrake = c.maxBrake; k.qy1 = c.qy1; k.qy2 = c.qy2;
    k.inv_m = c.inv_m; k.inv_jx = c.inv_jx; k.inv_jy = c.inv_jy; k.inv_jz = c.inv_jz;
    k.half_cf = c.half_cf; k.half_cr = c.half_cr;
    k.front = G == 4 ? q < 2 : q == 0;
    k.walks = group_walks(P);
    const double side = G == 4 && (q & 1) == 0 ? -1.0 : 1.0;  // a left corner's lane: minus
    k.mu = k.front ? P.muf : P.mur;
    k.mu_g = k.front ? c.mu_g[0] : c.mu_g[1];
    k.inv_mu = k.front ? c.inv_mu[0] : c.inv_mu[1];
    k.hrc = k.front ? P.hrcf : P.hrcr;
    k.inv_c = k.front ? P.d.inv_cf : P.d.inv_cr;
    k.track = side * (k.front ? P.cf : P.cr);
    k.arm = k.front ? P.a : -P.b;
}

// What the last step's record holds of this lane's corners (the chassis part on every lane).
template <int G>
struct X24g {
    static constexpr int N = 4 / G;
    double dOmega[N], dxt[N], fx[N], fy[N], fz[N], fxg[N], fyg[N], fzg[N], vgx[N], vgy[N], vsx[N], vsy[N];
    double My[N], engTor[N];
    double ls[N], us[N], vs[N], ws[N], dus[N], dvs[N], uu[N], vu[N], duu[N], dvu[N], dwu[N];
    double fxs[N], fys[N], fzs[N], mx[N], my[N];
    double dtheta, dphi, dpsi, dcrank;
};

// x and y from the new velocities at the yaw angle's sine and cosine, as position24 does.
template <int G>
LFDM_HD void move24g(S24g<G>& s, double sp, double cp, double dt) {
    s.x = s.x + (s.u * cp - s.v * sp) * dt;
    s.y = s.y + (s.u * sp + s.v * cp) * dt;
}

// step24 without its closing position update; `lag`: the previous step's position update comes first.
// The four angles' sines and cosines (pitch, roll, steering and, for the lagging update, yaw) are shared
// out: one angle per lane of four, two per lane of two.
template <bool NR, bool FULL, int G, class PS>
LFDM_HD void step24g(const PS& P, const Derived& u, const K24g<G>& k, S24g<G>& s, double steering, double throttle,
                     double braking, double dt, bool lag, X24g<G>* x) {
    constexpr int N = 4 / G;
    const TireP& t = P.tire;
    const double a = P.a, b = P.b;
    const double delta = P.nonLinearSteer ? map_y<false>(full_set(P).steer, steering) : steering * P.maxSteer;
    double sth, cth, sph, cph, sd, cd;
    if constexpr (G == 4) {
        double sa, ca;
        sincos_fast(s.q == 0 ? s.theta : s.q == 1 ? s.phi : s.q == 2 ? delta : s.psi, sa, ca);
        sth = group_value<4, 0>(sa); cth = group_value<4, 0>(ca);
        sph = group_value<4, 1>(sa); cph = group_value<4, 1>(ca);
        sd = group_value<4, 2>(sa); cd = group_value<4, 2>(ca);
        if (lag) move24g<G>(s, group_value<4, 3>(sa), group_value<4, 3>(ca), dt);
    } else {
        double sa, ca, sb, cb;
        sincos_fast(s.q == 0 ? s.theta : s.phi, sa, ca);
        sincos_fast(s.q == 0 ? delta : s.psi, sb, cb);
        sth = group_value<2, 0>(sa); cth = group_value<2, 0>(ca);
        sph = group_value<2, 1>(sa); cph = group_value<2, 1>(ca);
        sd = group_value<2, 0>(sb); cd = group_value<2, 0>(cb);
        if (lag) move24g<G>(s, group_value<2, 1>(sb), group_value<2, 1>(cb), dt);
    }
    // wheel loads from the compression, and the wheel speeds as the powertrain will read them: a tire off
    // the ground resets its own
    double fz[N], om[N], om4[4];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        fz[j] = s.xt[j] * t.kt;
        om[j] = fz[j] <= 0 ? 0 : s.omega[j];
    }
    group_tires<G>(om, om4);
    // computePowertrainRHS up to the wheels: nothing in it depends on this step's tire forces
    double shaft, dcrank, tf, tr;
    powertrain_group<G>(P, u, k.tqs, throttle, s.u, 0.25 * (om4[0] + om4[1] + om4[2] + om4[3]), s.q, k.walks, s.maps,
                        s.row, s.crank, s.gear, shaft, dcrank);
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
    // vehToSusTransform: strut-top velocities, strut length, unsprung-mass velocities
    const double vs = k.arm * s.wz + s.v;
    double us[N], ls[N], uu[N], vu[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const double tj = G == 4 || j == 1 ? k.track : -k.track;
        us[j] = (tj * s.wz / 2.) + s.u;
        ls[j] = k.lsi[j] - (s.xs[j] - k.xsi[j]);
        uu[j] = us[j] - ls[j] * s.wy;
        vu[j] = vs + ls[j] * s.wx;
    }
    // vehToTireTransform with last step's static radius, then computeTireRHS
    const double cc = cth * cph;
    const double rcc = frcp(cc);
    const double tand = fdiv(sd, cd);
    const double d = k.front ? tand : u.tan_delta_rear;
    double fx[N], fy[N], My[N], dOm[N];
    const double bt = k.maxBrake * braking;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const double vgx =
            cth * (uu[j] - s.wy * s.rStat[j]) + sth * (s.wu[j] * cph + sph * (s.wx * s.rStat[j] + vu[j]));
        const double vgy = cph * (vu[j] + s.wx * s.rStat[j]) - s.wu[j] * sph;
        const double vsy = vgy;
        const double vf = vgx * cd + vgy * sd;
        const double vsx = k.front ? vf : vgx;
        if (FULL) {
            x->vgx[j] = vgx; x->vgy[j] = vgy; x->vsx[j] = vsx; x->vsy[j] = vsy;
        }
        s.rStat[j] = (t.r0 - s.xt[j]) * rcc;
        if (fz[j] <= 0) {
            if (!NR) { s.xe[j] = 0; s.ye[j] = 0; }
            s.omega[j] = 0; s.xt[j] = 0; s.rStat[j] = t.r0; fz[j] = 0; fx[j] = 0; fy[j] = 0; My[j] = 0;
        } else if (!NR) {
            tmeasy_core<false>(t, u, k.qy1, k.qy2, 0.0, d, fz[j], s.rStat[j], vsx, vsy, s.xe[j], s.ye[j], s.omega[j],
                               s.xedot[j], s.yedot[j], fx[j], fy[j], My[j]);
        } else {
            tmeasy_nr_core<false>(t, u, k.qy1, k.qy2, 0.0, d, fz[j], s.rStat[j], vsx, vsy, s.omega[j], fx[j], fy[j],
                                  My[j]);
        }
        dOm[j] = u.inv_jw * (eng[j] + My[j] - sgn(s.omega[j]) * bt - fx[j] * s.rStat[j]);
        if (FULL) {
            x->dOmega[j] = dOm[j]; x->engTor[j] = eng[j]; x->fz[j] = fz[j]; x->My[j] = My[j];
        }
    }
    // Per corner: computeTireCompressionVelocity, tireToVehTransform, computeSusRHS (last step's fzd and dxs,
    // then the new dxs) and computeForcesThroughSus; the rear-right lateral force has no cos(theta)
    // factor in the reference (step24).  Each state is advanced as soon as nothing later reads its old
    // value, as in step24.
    double fyg[N], fxs[N], fys[N], fzs[N], my[N];
    const double dvs = k.arm * s.wzdot + s.vdot;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const double tj = G == 4 || j == 1 ? k.track : -k.track;
        const double dxt = k.vsz[j] - (cth * (s.wu[j] * cph + vu[j] * sph) - uu[j] * sth);
        if (!NR) {
            s.xe[j] = s.xe[j] + s.xedot[j] * dt;
            s.ye[j] = s.ye[j] + s.yedot[j] * dt;
        }
        s.xt[j] = s.xt[j] + dxt * dt;
        s.omega[j] = s.omega[j] + dOm[j] * dt;
        const double gx = fx[j] * cd - fy[j] * sd;
        const double gy = fx[j] * sd + fy[j] * cd;
        const double fxi = k.front ? gx : fx[j];
        const double fyi = k.front ? gy : fy[j];
        const double fxg = fxi * cth - fz[j] * sth;
        fyg[j] = fxi * sph * sth + fyi * cph + fz[j] * sph * cth;
        const double fzg = fxi * sth * cph - fyi * sph + fz[j] * cph * cth;
        const double dwu = k.inv_mu * (cph * (cth * (fz[j] - k.mu_g) + sth * fxi) - sph * fyi - s.fzd[j] -
                                       s.xs[j] * P.ks - s.dxs[j] * P.bs - k.mu * (vu[j] * s.wx - uu[j] * s.wy));
        const double dus = (tj * s.wzdot) / 2 + s.udot;
        const double ws = (-tj * s.wx / 2.) - (k.arm * s.wy) + s.w;
        const double duu = dus - (-s.dxs[j] * s.wy + ls[j] * s.wydot);
        const double dvu = dvs + (-s.dxs[j] * s.wx + ls[j] * s.wxdot);
        s.dxs[j] = -ws + s.wu[j];
        const bool rear_right = s.q == G - 1 && j == N - 1;
        const double ct = rear_right ? 1.0 : cth;
        fxs[j] = fxg + k.mu_g * sth - k.mu * duu + k.mu * s.wz * vu[j] - k.mu * s.wy * s.wu[j];
        fys[j] = fyg[j] - k.mu_g * sph * ct - k.mu * dvu + k.mu * s.wx * s.wu[j] - k.mu * s.wz * uu[j];
        fzs[j] = s.xs[j] * P.ks + s.dxs[j] * P.bs;
        my[j] = -(fxg * s.rStat[j] + fxs[j] * ls[j]);
        s.wu[j] = s.wu[j] + dwu * dt;
        s.xs[j] = s.xs[j] + s.dxs[j] * dt;
        if (FULL) {
            x->us[j] = us[j]; x->vs[j] = vs; x->ls[j] = ls[j]; x->uu[j] = uu[j]; x->vu[j] = vu[j]; x->dxt[j] = dxt;
            x->fx[j] = fxi; x->fy[j] = fyi; x->fxg[j] = fxg; x->fyg[j] = fyg[j]; x->fzg[j] = fzg;
            x->ws[j] = ws; x->dus[j] = dus; x->dvs[j] = dvs; x->duu[j] = duu; x->dvu[j] = dvu; x->dwu[j] = dwu;
            x->fxs[j] = fxs[j]; x->fys[j] = fys[j]; x->fzs[j] = fzs[j]; x->mx[j] = fys[j] * k.hrc; x->my[j] = my[j];
        }
    }
    if (P.tcbool) s.crank = s.crank + dcrank * dt;
    // the axle's jacking force, from this step's static radii
    {
        double fg0, fg1, fs0, fs1;  // fyg rStat and fys ls of the axle's left and right corner
        double y0, y1;              // fys
        if constexpr (G == 4) {
            const double pg = fyg[0] * s.rStat[0], ps = fys[0] * ls[0];
            fg0 = group_value<2, 0>(pg); fg1 = group_value<2, 1>(pg);
            fs0 = group_value<2, 0>(ps); fs1 = group_value<2, 1>(ps);
            y0 = group_value<2, 0>(fys[0]); y1 = group_value<2, 1>(fys[0]);
        } else {
            fg0 = fyg[0] * s.rStat[0]; fg1 = fyg[1] * s.rStat[1];
            fs0 = fys[0] * ls[0]; fs1 = fys[1] * ls[1];
            y0 = fys[0]; y1 = fys[1];
        }
        const double jk = fg1 + fs1 + fg0 + fs0 - (y1 + y0) * k.hrc;
        const double fd = jk * k.inv_c;
        if constexpr (G == 4) {
            s.fzd[0] = (s.q & 1) ? fd : -fd;
        } else {
            s.fzd[1] = fd;
            s.fzd[0] = -fd;
        }
    }
    double fxs4[4], fys4[4], fzs4[4], my4[4], fzd4[4];
    group_tires<G>(fxs, fxs4);
    group_tires<G>(fys, fys4);
    group_tires<G>(fzs, fzs4);
    group_tires<G>(my, my4);
    group_tires<G>(s.fzd, fzd4);
    // computeVehicleRHS, the sums in the reference's order
    const double sfxs = fxs4[0] + fxs4[1] + fxs4[2] + fxs4[3];
    const double sfys = fys4[0] + fys4[1] + fys4[2] + fys4[3];
    const double sfzs = fzs4[0] + fzs4[1] + fzs4[2] + fzs4[3];
    const double smx = fys4[0] * P.hrcf + fys4[1] * P.hrcf + fys4[2] * P.hrcr + fys4[3] * P.hrcr;
    const double smy = my4[0] + my4[1] + my4[2] + my4[3];
    const double tF = (fzs4[0] - fzs4[1]) * k.half_cf, sF = fzs4[0] + fzs4[1];
    const double tA = (fys4[0] + fys4[1]) * a, tC = (-fxs4[0] + fxs4[1]) * k.half_cf;
    const double tR = (fzs4[2] - fzs4[3]) * k.half_cr, sR = fzs4[2] + fzs4[3];
    const double tB = (fys4[2] + fys4[3]) * b, tD = (-fxs4[2] + fxs4[3]) * k.half_cr;
    const double udot = s.wz * s.v - s.wy * s.w + k.inv_m * sfxs + kG * sth;
    const double vdot = s.wx * s.w - s.wz * s.u + k.inv_m * sfys - kG * sph * cth;
    const double wdot = s.wy * s.u - s.wx * s.v + k.inv_m * (sfzs + fzd4[0] + fzd4[1] + fzd4[2] + fzd4[3]) -
                        kG * cph * cth;
    const double wxdot = k.inv_jx * (smx + tF + tR);
    const double wydot = k.inv_jy * (smy + sR * b - sF * a);
    const double wzdot = k.inv_jz * (0.0 + tA - tB + tC + tD);
    s.u = s.u + udot * dt;
    s.v = s.v + vdot * dt;
    s.w = s.w + wdot * dt;
    s.wx = s.wx + wxdot * dt;
    s.wy = s.wy + wydot * dt;
    s.wz = s.wz + wzdot * dt;
    // Euler-angle rates at the step's (old) theta and phi
    const double rcth = cph * rcc;
    const double tth = sth * rcth;
    const double dtheta = s.wy * cph - s.wz * sph;
    const double dpsi = (s.wy * sph * rcth) + (s.wz * cph * rcth);
    const double dphi = s.wx + s.wy * sph * tth + s.wz * cph * tth;
    s.theta = s.theta + dtheta * dt;
    s.psi = s.psi + dpsi * dt;
    s.phi = s.phi + dphi * dt;
    s.udot = udot;
    s.vdot = vdot;
    s.wdot = wdot;
    s.wxdot = wxdot;
    s.wydot = wydot;
    s.wzdot = wzdot;
    if (FULL) {
        x->dtheta = dtheta;
        x->dphi = dphi;
        x->dpsi = dpsi;
        x->dcrank = dcrank;
    }
}

}  // namespace dev
}  // namespace lfdm
