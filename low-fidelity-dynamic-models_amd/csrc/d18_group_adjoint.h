// The adjoint of the 18-DOF step (d18_adjoint.h) on a group of G lanes (2: an axle per lane, 4: a tire per
// lane), from a tape that holds the step's tire outputs.  Same operations in the same order as step18_adj
// for every value, so the same bits: the tires' reverse sweeps and map lookups are shared out, the chassis
// and the adjoints of the per-vehicle constants are on every lane.
#pragma once
#include "d18_adjoint_lanes.h"
#include "d18_group.h"

namespace lfdm {
namespace dev {

// Adjoint of one lane's carried state: its own tires' and the chassis's.
template <int G>
struct S18gb {
    static constexpr int N = 4 / G;
    double xe[N], ye[N], xedot[N], yedot[N], omega[N];
    double x, y, u, v, psi, wz, phi, wx, udot, vdot, crank;
};

template <int G>
LFDM_HD void s18gb_zero(S18gb<G>& b) {
#pragma unroll
    for (int j = 0; j < 4 / G; ++j) b.xe[j] = b.ye[j] = b.xedot[j] = b.yedot[j] = b.omega[j] = 0.0;
    b.x = b.y = b.u = b.v = b.psi = b.wz = b.phi = b.wx = b.udot = b.vdot = b.crank = 0.0;
}

// What the tape holds of one step: the state before it and its tire outputs.
template <int G>
struct Tape18g {
    static constexpr int N = 4 / G;
    double xe[N], ye[N], omega[N];
    double u, v, psi, wz, phi, wx, udot, vdot, crank;
    int gear;
    TireOut18g<G> to;
};

// The sweep's places on the maps and the row of the gear it last met.
template <int G>
struct Sweep18g {
    Walks<G> maps;
    GearRow row;
    int gear;
};

template <int G>
LFDM_HD void sweep18g_init(const PSet& P, const MapXY* tab, double tqs, int q, Sweep18g<G>& w) {
    walks_init<G>(P, tab, tqs, q, w.maps);
    w.gear = 0;
    gear_row(P, 0, w.row);
}

// map_y_slope by the walk: the value at x and the slope of its segment (0 where the map clamps); scaled is
// the value with the ordinates' factor applied first, as map_y_scaled forms it.
LFDM_HD double walk_slope(Walk& w, MapXY L, MapXY R, double x, double& slope, double& scaled) {
    walk_to(w, L, R, x);
    const bool below = x <= w.first.x, above = x >= w.last.x;
    const double m = fdiv(R.y - L.y, R.x - L.x);
    const double mbar = fdiv(x - L.x, R.x - L.x);
    const double y = L.y + mbar * (R.y - L.y);
    const double ly = L.y * w.scale, ry = R.y * w.scale;
    const double ys = ly + mbar * (ry - ly);
    slope = below || above ? 0.0 : m;
    scaled = below ? w.first.y * w.scale : (above ? w.last.y * w.scale : ys);
    return below ? w.first.y : (above ? w.last.y : y);
}

// powertrain4_adj: om4 the four wheel speeds after the tires' resets; fx, rStat this lane's; dOmb its bars of
// the wheel accelerations (in).  Returns this lane's bars of omega, fx, rStat and My (omb accumulates) and,
// on every lane, those of crank, throttle, braking, tqs and maxBrake.
template <int G>
LFDM_HD void powertrain_group_adj(const PSet& P, const Derived& u, const K18& c, const K18g<G>& k, int q, Sweep18g<G>& w,
                                  double throttle, double braking, double vel_u, double crank, int gear,
                                  const double* om4, const double* fx, const double* rStat, const double* dOmb,
                                  double dcrankb, double crank_outb, double* omb, double* fxb, double* rStatb,
                                  double* Myb, double& crankb, double& thrb, double& brkb, double& tqsb,
                                  double& maxBrakeb) {
    constexpr int N = 4 / G;
    const double tqs = c.tqs, maxBrake = c.maxBrake;
    if (gear != w.gear) {
        w.gear = gear;
        gear_row(P, gear, w.row);
    }
    const MapXY La = w.maps.a.e[w.maps.a.r - 1], Ra = w.maps.a.e[w.maps.a.r];
    MapXY Lb{}, Rb{};
    if constexpr (G == 2) {
        Lb = w.maps.b.e[w.maps.b.r - 1];
        Rb = w.maps.b.e[w.maps.b.r];
    }
    const double gr = w.row.ratio;
    const double osum = om4[0] + om4[1] + om4[2] + om4[3];
    // ---- forward recompute ----
    const double omega_out = fdiv_by(0.25 * osum, gr, w.row.rcp);
    const double omega_in = crank;
    double sr0 = 0, sr = 0;
    bool active = false, rev = false;
    double w_dt = crank;  // crank speed the drive torque is evaluated at
    if (P.tcbool) {
        const double quot = fdiv(omega_out, omega_in);
        active = !(omega_out < 1e-9 || omega_in < 1e-9);
        sr0 = active ? quot : 0.0;
        rev = sr0 > 1.;
        sr = rev ? 1. - (sr0 - 1.) : sr0;
        if (sr < 0) {
            sr = 0;
            active = false;
        }
    } else {
        w_dt = omega_out;
    }
    double cf = 1, cfs = 0, tr = 1, trs = 0, Tw, Ts, Ls, drive = 0;
    if (!k.walks) {  // maps that do not ascend are scanned
        if (P.tcbool) {
            cf = map_y_slope(P.cfmap, sr, cfs);
            tr = map_y_slope(P.trmap, sr, trs);
        } else {
            drive = drive_torque<false>(P, tqs, throttle, w_dt);
        }
        Tw = map_y_slope(P.torque, w_dt, Ts);
        map_y_slope(P.losses, w_dt, Ls);
    } else if constexpr (G == 4) {
        double m, ys;
        const double y = walk_slope(w.maps.a, La, Ra, q < 2 ? sr : w_dt, m, ys);
        cf = group_value<4, kMapCf>(y);
        tr = group_value<4, kMapTr>(y);
        Tw = group_value<4, kMapTorque>(y);
        cfs = group_value<4, kMapCf>(m);
        trs = group_value<4, kMapTr>(m);
        Ts = group_value<4, kMapTorque>(m);
        Ls = group_value<4, kMapLosses>(m);
        drive = group_value<4, kMapTorque>(ys) * throttle + group_value<4, kMapLosses>(y);
    } else {
        double ma, mb, ys;
        const double ya = walk_slope(w.maps.a, La, Ra, sr, ma, ys), yb = walk_slope(w.maps.b, Lb, Rb, w_dt, mb, ys);
        cf = group_value<2, 0>(ya);
        tr = group_value<2, 1>(ya);
        Tw = group_value<2, 0>(yb);
        cfs = group_value<2, 0>(ma);
        trs = group_value<2, 1>(ma);
        Ts = group_value<2, 0>(mb);
        Ls = group_value<2, 1>(mb);
        drive = group_value<2, 0>(ys) * throttle + group_value<2, 1>(yb);
    }
    double torque_t, torque_in = 0, qc = 0;
    if (P.tcbool) {
        qc = fdiv(omega_in, cf);
        torque_in = -(qc * qc);
        torque_in = rev ? -torque_in : torque_in;
        const double torque_out = rev ? -torque_in : -tr * torque_in;
        torque_t = fdiv_by(torque_out, gr, w.row.rcp);
    } else {
        torque_t = fdiv_by(drive, gr, w.row.rcp);
    }
    const bool clip = vel_u < 1e-9 && torque_t < 0;
    torque_t = clip ? 0.0 : torque_t;
    double tf, trr;
    axle_torques(P, torque_t, tf, trr);
    // ---- reverse ----
    double engb[N], bs[N], bs4[4], engb_l, engb_r;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const double cm = dOmb[j] * u.inv_jw;
        const int i = G == 4 ? 0 : j;
        engb[j] = cm;
        Myb[j] = cm;
        const double own = G == 4 ? (k.front ? ((q & 1) ? om4[1] : om4[0]) : ((q & 1) ? om4[3] : om4[2]))
                                  : (k.front ? om4[i] : om4[2 + i]);
        bs[j] = cm * sgn(own);
        fxb[j] = -(cm * rStat[j]);
        rStatb[j] = -(cm * fx[j]);
    }
    group_tires<G>(bs, bs4);
    double btb = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) btb -= bs4[i];
    maxBrakeb = btb * braking;
    brkb = btb * maxBrake;
    if constexpr (G == 4) {
        engb_l = group_value<2, 0>(engb[0]);
        engb_r = group_value<2, 1>(engb[0]);
    } else {
        engb_l = engb[0];
        engb_r = engb[1];
    }
    double axb = 0, lb = 0, rb = 0;
    diff_split_adj(k.front ? tf : trr, k.front ? om4[0] : om4[2], k.front ? om4[1] : om4[3], engb_l, engb_r, axb, lb, rb);
    const double tfb = group_value<G, 0>(axb), trrb = group_value<G, G / 2>(axb);
    if constexpr (G == 4) {
        omb[0] += (q & 1) ? rb : lb;
    } else {
        omb[0] += lb;
        omb[1] += rb;
    }
    double ttb = P.driveType ? 0.5 * (tfb + trrb) : P.whichWheels ? trrb : tfb;
    ttb = clip ? 0.0 : ttb;
    // drive torque at w_dt: tqs * T(w) * throttle + L(w)
    const double rgr = frcp(gr);
    if (P.tcbool) {
        double toutb = ttb * rgr;
        double tinb = rev ? -toutb : -tr * toutb;
        const double trb = rev ? 0.0 : -toutb * torque_in;
        // dcrank = inv_ci (DT + torque_in)
        const double DTb = dcrankb * u.inv_ci;
        tinb += dcrankb * u.inv_ci;
        tqsb = DTb * Tw * throttle;
        thrb = DTb * tqs * Tw;
        crankb = DTb * (tqs * throttle * Ts + Ls);
        // torque_in = -q^2 (negated when reversed)
        const double qb = tinb * (rev ? 2.0 * qc : -2.0 * qc);
        const double qbr = fdiv(qb, cf);
        double omega_inb = qbr;
        const double cfb = -qbr * qc;
        const double srb = cfb * cfs + trb * trs;
        if (active) {
            const double sr0b = rev ? -srb : srb;
            const double omega_outb = fdiv(sr0b, omega_in);
            omega_inb -= omega_outb * sr0;
            const double ob = omega_outb * 0.25 * rgr;
#pragma unroll
            for (int j = 0; j < N; ++j) omb[j] += ob;
        }
        crankb += omega_inb;
    } else {
        const double DTb = ttb * rgr;
        tqsb = DTb * Tw * throttle;
        thrb = DTb * tqs * Tw;
        crankb = 0.0;
        const double wb = (crank_outb + DTb * (tqs * throttle * Ts + Ls)) * 0.25 * rgr;
#pragma unroll
        for (int j = 0; j < N; ++j) omb[j] += wb;
    }
}

// step18_adj from the tape: sb in: adjoint of the state after the step, out: of the state before it.
template <int G>
LFDM_HD void step18g_adj(const PSet& P, const Derived& u, const K18& c, const K18g<G>& k, const Tape18g<G>& s0, int q,
                         Sweep18g<G>& w, double steering, double throttle, double braking, double dt, S18gb<G>& sb,
                         double& steerb, double& thrb, double& brkb, K18b& kb) {
    constexpr int N = 4 / G;
    const TireP& t = P.tire;
    // ================= forward recompute =================
    const double lat = s0.vdot + s0.wz * s0.u;
    double fzr[N], fz[N], om[N], om4[4];
    loads18g<G>(c, k, lat, s0.phi, s0.wx, s0.udot, s0.wz, s0.v, fzr);
#pragma unroll
    for (int j = 0; j < N; ++j) {
        fz[j] = fzr[j] > 0. ? fzr[j] : 0.;
        om[j] = fz[j] <= 0 ? 0 : s0.omega[j];
    }
    group_tires<G>(om, om4);
    // one lane takes the steering angle's sine and cosine while another takes the yaw angle's
    double sa, ca;
    sincos_fast((q & 1) ? s0.psi : steering * P.maxSteer, sa, ca);
    const double sd = group_value<G, 0>(sa), cd = group_value<G, 0>(ca);
    const double sp = group_value<G, 1>(sa), cp = group_value<G, 1>(ca);
    double vsx[N];
    const double vsy = patch18g<G>(k, s0.u, s0.v, s0.wz, sd, cd, vsx);
    double fx4[4], fy4[4], gfx[4], gfy[4];
    group_tires<G>(s0.to.fx, fx4);
    group_tires<G>(s0.to.fy, fy4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        gfx[i] = i < 2 ? fx4[i] * cd - fy4[i] * sd : fx4[i];
        gfy[i] = i < 2 ? fx4[i] * sd + fy4[i] * cd : fy4[i];
    }
    // ================= reverse =================
    const S18gb<G> o = sb;
    s18gb_zero<G>(sb);
    double dOmb[N], omb[N], xedotb[N], yedotb[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        dOmb[j] = o.omega[j] * dt;
        omb[j] = 0;
        xedotb[j] = o.xe[j] * dt + o.xedot[j];
        yedotb[j] = o.ye[j] * dt + o.yedot[j];
    }
    if (P.tcbool) sb.crank += o.crank;
    double fxpb[N], rStatb[N], Myb[N], crankb, thb, bkb, tqsb, mbb;
    powertrain_group_adj<G>(P, u, c, k, q, w, throttle, braking, s0.u, s0.crank, s0.gear, om4, s0.to.fx, s0.to.rStat, dOmb,
                            P.tcbool ? o.crank * dt : 0.0, P.tcbool ? 0.0 : o.crank, omb, fxpb, rStatb, Myb, crankb, thb,
                            bkb, tqsb, mbb);
    double gfxb[4], gfyb[4];
    chassis18_adj(P, u, c, s0, gfx, gfy, sp, cp, dt, o, sb, kb, gfxb, gfyb);
    // ---- tireToVehTransform (front tires rotated by delta) ----
    double sdb = 0, cdb = 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        sdb += -gfxb[i] * fy4[i] + gfyb[i] * fx4[i];
        cdb += gfxb[i] * fx4[i] + gfyb[i] * fy4[i];
    }
    thrb += thb;
    brkb += bkb;
    kb.tqs += tqsb;
    kb.maxBrake += mbb;
    sb.crank += crankb;
    // ---- this lane's tires ----
    const double tand = fdiv(sd, cd);
    const double d = k.front ? tand : u.tan_delta_rear;
    double rb[N], vsxb[N], vsyb[N], db[N], q1b[N], q2b[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        rb[j] = vsxb[j] = vsyb[j] = db[j] = q1b[j] = q2b[j] = 0;
        if (fz[j] <= 0) {
            // reset: xe, ye, omega become 0 (their incoming bars stop here); xedot, yedot pass through
            sb.xedot[j] += xedotb[j];
            sb.yedot[j] += yedotb[j];
            continue;
        }
        // the forces' bars in the tire's axes
        double gx, gy;
        if constexpr (G == 4) {
            gx = k.front ? ((q & 1) ? gfxb[1] : gfxb[0]) : ((q & 1) ? gfxb[3] : gfxb[2]);
            gy = k.front ? ((q & 1) ? gfyb[1] : gfyb[0]) : ((q & 1) ? gfyb[3] : gfyb[2]);
        } else {
            gx = k.front ? gfxb[j] : gfxb[2 + j];
            gy = k.front ? gfyb[j] : gfyb[2 + j];
        }
        const double fxr = gx * cd + gy * sd, fyr = -gx * sd + gy * cd;
        TireBars tb;
        tb.xedot = xedotb[j];
        tb.yedot = yedotb[j];
        tb.fx = (k.front ? fxr : gx) + fxpb[j];
        tb.fy = k.front ? fyr : gy;
        tb.My = Myb[j];
        tb.rStat = rStatb[j];
        tb.fz = tb.vsx = tb.vsy = tb.delta = tb.xe = tb.ye = tb.omega = tb.qy1 = tb.qy2 = 0.0;
        tire_tmeasy_adj(t, u, c.qy1, c.qy2, d, fz[j], vsx[j], vsy, s0.xe[j], s0.ye[j], s0.omega[j], tb);
        sb.xe[j] += o.xe[j] + tb.xe;
        sb.ye[j] += o.ye[j] + tb.ye;
        sb.omega[j] += (o.omega[j] + omb[j]) + tb.omega;
        rb[j] = fzr[j] > 0. ? tb.fz : 0.;
        vsxb[j] = tb.vsx;
        vsyb[j] = tb.vsy;
        db[j] = tb.delta;
        q1b[j] = tb.qy1;
        q2b[j] = tb.qy2;
    }
    double rb4[4], vsxb4[4], vsyb4[4], db4[4], q4[4];
    group_tires<G>(rb, rb4);
    group_tires<G>(vsxb, vsxb4);
    group_tires<G>(vsyb, vsyb4);
    group_tires<G>(db, db4);
    const double deltab = db4[0] + db4[1];
    group_tires<G>(q1b, q4);
#pragma unroll
    for (int i = 0; i < 4; ++i) kb.qy1 += q4[i];
    group_tires<G>(q2b, q4);
#pragma unroll
    for (int i = 0; i < 4; ++i) kb.qy2 += q4[i];
    body18_adj(P, u, c, s0, lat, sd, cd, s0.v + s0.wz * P.a, vsxb4, vsyb4, rb4, deltab, sdb, cdb, sb, steerb, kb);
}

// ---- per-lane bodies of the group kernels (as d18_adjoint_lanes.h's, same buffers) ----

template <int G>
LFDM_HD void tape_put_state_g(const S18g<G>& s, double* p) {
    constexpr int N = 4 / G;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int i = N * s.q + j;
        p[(0 + i) * kWave] = s.xe[j];
        p[(4 + i) * kWave] = s.ye[j];
        p[(8 + i) * kWave] = s.omega[j];
    }
    if (s.q != 0) return;
    const double v[9] = {s.u, s.v, s.psi, s.wz, s.phi, s.wx, s.udot, s.vdot, s.crank};
#pragma unroll
    for (int j = 0; j < 9; ++j) p[(12 + j) * kWave] = v[j];
    p[21 * kWave] = (double)s.gear;
}

template <int G>
LFDM_HD void tape_put_tires_g(const TireOut18g<G>& t, int q, double* p) {
    constexpr int N = 4 / G;
    p += (size_t)kTapeState * kWave;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int i = N * q + j;
        p[(0 + i) * kWave] = t.fx[j];
        p[(4 + i) * kWave] = t.fy[j];
        p[(8 + i) * kWave] = t.My[j];
        p[(12 + i) * kWave] = t.rStat[j];
    }
}

template <int G>
LFDM_HD void tape_get_g(const double* p, int q, Tape18g<G>& s) {
    constexpr int N = 4 / G;
    const double* t = p + (size_t)kTapeState * kWave;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int i = N * q + j;
        s.xe[j] = p[(0 + i) * kWave];
        s.ye[j] = p[(4 + i) * kWave];
        s.omega[j] = p[(8 + i) * kWave];
        s.to.fx[j] = t[(0 + i) * kWave];
        s.to.fy[j] = t[(4 + i) * kWave];
        s.to.My[j] = t[(8 + i) * kWave];
        s.to.rStat[j] = t[(12 + i) * kWave];
    }
    s.u = p[12 * kWave]; s.v = p[13 * kWave]; s.psi = p[14 * kWave]; s.wz = p[15 * kWave]; s.phi = p[16 * kWave];
    s.wx = p[17 * kWave]; s.udot = p[18 * kWave]; s.vdot = p[19 * kWave]; s.crank = p[20 * kWave];
    s.gear = (int)p[21 * kWave];
}

// A lane's part of a checkpoint (pack's rows).
template <int G>
LFDM_HD void pack_g(const S18g<G>& s, double* p, size_t S) {
    constexpr int N = 4 / G;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int i = N * s.q + j;
        p[(0 + i) * S] = s.xe[j];
        p[(4 + i) * S] = s.ye[j];
        p[(8 + i) * S] = s.xedot[j];
        p[(12 + i) * S] = s.yedot[j];
        p[(16 + i) * S] = s.omega[j];
    }
    if (s.q != 0) return;
    const double v[11] = {s.x, s.y, s.u, s.v, s.psi, s.wz, s.phi, s.wx, s.udot, s.vdot, s.crank};
#pragma unroll
    for (int j = 0; j < 11; ++j) p[(20 + j) * S] = v[j];
    p[31 * S] = (double)s.gear;
}

// Carried state of one slot from the SoA record array (TMeasy layout), this lane's tires.
template <int G>
LFDM_HD void load_record_g(const double* st, size_t S, int slot, S18g<G>& s) {
    constexpr int N = 4 / G;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int i = N * s.q + j;
        s.xe[j] = st[(size_t)(i * 15 + 0) * S + slot];
        s.ye[j] = st[(size_t)(i * 15 + 1) * S + slot];
        s.xedot[j] = st[(size_t)(i * 15 + 2) * S + slot];
        s.yedot[j] = st[(size_t)(i * 15 + 3) * S + slot];
        s.omega[j] = st[(size_t)(i * 15 + 4) * S + slot];
    }
    const double* v = st + (size_t)60 * S + slot;
    s.x = v[0 * S]; s.y = v[1 * S]; s.u = v[2 * S]; s.v = v[3 * S]; s.psi = v[4 * S]; s.wz = v[5 * S];
    s.phi = v[6 * S]; s.wx = v[7 * S]; s.udot = v[8 * S]; s.vdot = v[9 * S]; s.crank = v[12 * S];
    s.gear = (int)v[14 * S];
}

// adj_forward_lane on a group.  A step's position update comes with the next step's angles, so the positions
// of step j are written by step j + 1 (the last step's after the loop).
// HOT: the set's parameters in registers (HotSet).  On four lanes, which have the registers, the controls are
// loaded a step ahead of their use.  Per step 2.95 -> 2.83 us (1,000 vehicles), 3.30 -> 3.13 (16,384), 4.90 -> 4.62
// (32,768, two wavefronts per SIMD: controls only).  The reverse sweep has no room for either: with HotSet 6.33 ->
// 6.86 (1,000), with the next tape row held 6.53.
template <int G, bool HOT>
LFDM_HD void adj_forward_group(const AdjLaunch& L, int slot, int q, const PSet& P, const MapXY* tab) {
    const size_t S = (size_t)L.S, N = (size_t)L.n_user;
    S18g<G> s;
    s.q = q;
    load_record_g<G>(L.state, S, slot, s);
    K18 c;
    load_k(P, L.ovr + slot, S, c);
    K18g<G> k;
    k18g_init<G>(P, c, q, k);
    walks_init<G>(P, tab, c.tqs, q, s.maps);
    gear_row(P, s.gear, s.row);
    Params<HOT> set;
    set.init(P);
    const auto& h = set.of(P);
    const int user = L.slot_user[slot];
    const int uv = user >= 0 ? user : 0;
    const bool writes = user >= 0 && q == 0;
    const int jt = L.fwd_tape_lo * L.K < L.nsteps ? L.fwd_tape_lo * L.K : L.nsteps;
    int seg = 0, jj = 0;  // segment of step j and the step's index in it
    constexpr bool kAhead = G == 4;
    const double* ctl = L.ctrl + uv;
    double next[3] = {ctl[0], ctl[N], ctl[2 * N]};
    for (int j = 0; j < L.nsteps; ++j) {
        const double steering = next[0], throttle = next[1], braking = next[2];
        if (kAhead && j + 1 < L.nsteps) {
            ctl += 3 * N;
            next[0] = ctl[0]; next[1] = ctl[N]; next[2] = ctl[2 * N];
        }
        double sd, cd;
        angles18g<G>(h, s, steering, L.dt, j > 0, sd, cd);
        if (writes && j > 0) {
            L.xy[(size_t)(j - 1) * 2 * N + user] = s.x;
            L.xy[((size_t)(j - 1) * 2 + 1) * N + user] = s.y;
        }
        if (jj == 0) pack_g<G>(s, L.ckpt + (size_t)seg * kCarried * S + slot, S);
        if (j < jt) {
            step18g<false, false, G>(h, h.d, c, k, s, sd, cd, throttle, braking, L.dt, nullptr);
        } else {
            double* row = tape_row(L, seg - L.fwd_tape_lo, jj, slot);
            tape_put_state_g<G>(s, row);
            TireOut18g<G> to;
            step18g<false, false, G, true>(h, h.d, c, k, s, sd, cd, throttle, braking, L.dt, nullptr, &to);
            tape_put_tires_g<G>(to, q, row);
        }
        if (++jj == L.K) {
            jj = 0;
            ++seg;
        }
        if (!kAhead && j + 1 < L.nsteps) {
            ctl += 3 * N;
            next[0] = ctl[0]; next[1] = ctl[N]; next[2] = ctl[2 * N];
        }
    }
    double sp, cp;
    sincos_fast(s.psi, sp, cp);
    move18g<G>(s, sp, cp, L.dt);
    if (writes) {
        L.xy[(size_t)(L.nsteps - 1) * 2 * N + user] = s.x;
        L.xy[((size_t)(L.nsteps - 1) * 2 + 1) * N + user] = s.y;
    }
}

// A lane's part of the running adjoints between reverse launches (store_carry's rows; the chassis's and the
// constants' from lane 0).
template <int G>
LFDM_HD void store_carry_g(const S18gb<G>& l, const K18b& kb, int q, double* p, size_t S) {
    constexpr int N = 4 / G;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int i = N * q + j;
        p[(0 + i) * S] = l.xe[j];
        p[(4 + i) * S] = l.ye[j];
        p[(8 + i) * S] = l.xedot[j];
        p[(12 + i) * S] = l.yedot[j];
        p[(16 + i) * S] = l.omega[j];
    }
    if (q != 0) return;
    S18b b;
    s18b_zero(b);
    b.x = l.x; b.y = l.y; b.u = l.u; b.v = l.v; b.psi = l.psi; b.wz = l.wz; b.phi = l.phi; b.wx = l.wx;
    b.udot = l.udot; b.vdot = l.vdot; b.crank = l.crank;
    store_carry_body(b, kb, p, S);
}

template <int G>
LFDM_HD void load_carry_g(const double* p, size_t S, int q, S18gb<G>& l, K18b& kb) {
    constexpr int N = 4 / G;
    S18b b;
    load_carry(p, S, b, kb);
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int i = N * q + j;
        l.xe[j] = p[(0 + i) * S];
        l.ye[j] = p[(4 + i) * S];
        l.xedot[j] = p[(8 + i) * S];
        l.yedot[j] = p[(12 + i) * S];
        l.omega[j] = p[(16 + i) * S];
    }
    l.x = b.x; l.y = b.y; l.u = b.u; l.v = b.v; l.psi = b.psi; l.wz = b.wz; l.phi = b.phi; l.wx = b.wx;
    l.udot = b.udot; l.vdot = b.vdot; l.crank = b.crank;
}

// Storage of T lanes' constants and the adjoints of them.  Every lane adds every contribution to its own copy
// of the adjoints: in one copy per vehicle an addition would count once only while the group's lanes load and
// store it in step.  The constants, which each lane writes before it reads them, all the same values, need one.
template <int G, int T>
struct ReverseStore {
    K18 c[T / G];
    K18b kb[T];
    LFDM_HD K18& constants(int lane) { return c[lane / G]; }
    LFDM_HD K18b& adjoints(int lane) { return kb[lane]; }
};

// adj_reverse_lane on a group; c, kb: this lane's of a ReverseStore.
template <int G>
LFDM_HD void adj_reverse_group(const AdjLaunch& L, int slot, int q, const PSet& P, const MapXY* tab, K18& c, K18b& kb) {
    const size_t S = (size_t)L.S, N = (size_t)L.n_user;
    const int nseg = (L.nsteps + L.K - 1) / L.K;
    load_k(P, L.ovr + slot, S, c);
    K18g<G> k;
    k18g_init<G>(P, c, q, k);
    Sweep18g<G> w;
    sweep18g_init<G>(P, tab, c.tqs, q, w);
    const int user = L.slot_user[slot];
    const int uv = user >= 0 ? user : 0;
    S18gb<G> lam;
    if (L.seg_hi >= nseg) {
        s18gb_zero<G>(lam);
        k18b_zero(kb);
    } else {
        load_carry_g<G>(L.carry + slot, S, q, lam, kb);
    }
    for (int seg = L.seg_hi - 1; seg >= L.seg_lo; --seg) {
        const int j0 = seg * L.K;
        const int j1 = (L.nsteps < j0 + L.K ? L.nsteps : j0 + L.K);
        for (int j = j1 - 1; j >= j0; --j) {
            LFDM_RELOAD_MEMORY();
            Tape18g<G> s;
            tape_get_g<G>(tape_row(L, seg - L.seg_lo, j - j0, slot), q, s);
            lam.x += L.xy_bar[(size_t)j * 2 * N + uv];
            lam.y += L.xy_bar[((size_t)j * 2 + 1) * N + uv];
            const double* ctl = L.ctrl + (size_t)j * 3 * N + uv;
            double sb = 0, tb = 0, bb = 0;
            step18g_adj<G>(P, P.d, c, k, s, q, w, ctl[0], ctl[N], ctl[2 * N], L.dt, lam, sb, tb, bb, kb);
            if (user >= 0 && q == 0) {
                double* cb = L.ctrl_bar + (size_t)j * 3 * N + user;
                cb[0] = sb;
                cb[N] = tb;
                cb[2 * N] = bb;
            }
        }
    }
    if (L.seg_lo > 0) {
        store_carry_g<G>(lam, kb, q, L.carry + slot, S);
        return;
    }
    if (user < 0) return;
    // adjoint of the initial record, each lane its own tires (15 fields each) and lane 0 the vehicle block
    constexpr int NT = 4 / G;
    double* g = L.state_bar + user;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int i = NT * q + j;
        const double f[5] = {lam.xe[j], lam.ye[j], lam.xedot[j], lam.yedot[j], lam.omega[j]};
#pragma unroll
        for (int m = 0; m < 15; ++m) g[(size_t)(15 * i + m) * N] = m < 5 ? f[m < 5 ? m : 0] : 0.0;
    }
    if (q != 0) return;
    const double v[15] = {lam.x, lam.y, lam.u, lam.v, lam.psi, lam.wz, lam.phi, lam.wx, lam.udot, lam.vdot,
                          0.0,   0.0,   lam.crank, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < 15; ++j) g[(size_t)(60 + j) * N] = v[j];
    double pb[7] = {0, 0, 0, 0, 0, 0, 0};
    k18_init_adj(P, c, kb, pb);
#pragma unroll
    for (int i = 0; i < 7; ++i) L.param_bar[i * N + user] = pb[i];
}

}  // namespace dev
}  // namespace lfdm
