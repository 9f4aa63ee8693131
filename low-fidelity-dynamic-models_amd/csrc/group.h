// One vehicle on a group of neighbouring lanes: the exchange of values inside a group.
//
// The group steps (d11_group.h, d18_group.h, d24_group.h) give every lane of a group its own tires (one
// or two of a vehicle's four; one of the 11-DOF model's two) and let all of them run the chassis and the
// powertrain, each on the same values and with the operations and the order of the one-lane step, so a
// vehicle's results have the same bits whichever kernel ran it.  Values cross lanes through quad
// permutes (v_mov_b32_dpp quad_perm: two VALU moves per double, no LDS and no wait); a group is 2 or 4
// lanes aligned to its size, so it never straddles a quad.
#pragma once
#include "dev_tire.h"

namespace lfdm {
namespace dev {

#if !defined(__HIP_DEVICE_COMPILE__)
// Host builds run a vehicle's lanes as threads that meet at every exchange; the caller installs the
// exchange, which returns the v of lane q of this lane's group of g.
inline thread_local double (*host_group_exchange)(double v, int g, int q) = nullptr;
#endif

// The value lane Q of this lane's group of G holds in v.  Every lane of the group must be active.
template <int G, int Q>
LFDM_HD double group_value(double v) {
    static_assert((G == 2 || G == 4) && Q < G, "groups of 2 or 4 lanes");
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int perm = G == 4 ? Q | Q << 2 | Q << 4 | Q << 6 : Q | Q << 2 | (2 + Q) << 4 | (2 + Q) << 6;
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, perm, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), perm, 0xf, 0xf, true);
    return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
#else
    return host_group_exchange(v, G, Q);
#endif
}

// The values of a vehicle's four tires (LF RF LR RR) from its lanes' own, v[4 / G] each: lane q of a
// group holds the tires 4 / G * q onwards.
template <int G>
LFDM_HD void group_tires(const double* v, double* all) {
    if constexpr (G == 4) {
        all[0] = group_value<4, 0>(v[0]);
        all[1] = group_value<4, 1>(v[0]);
        all[2] = group_value<4, 2>(v[0]);
        all[3] = group_value<4, 3>(v[0]);
    } else {
        all[0] = group_value<2, 0>(v[0]);
        all[1] = group_value<2, 0>(v[1]);
        all[2] = group_value<2, 1>(v[0]);
        all[3] = group_value<2, 1>(v[1]);
    }
}

// The powertrain's four map lookups of a step (capacity factor and torque ratio at the converter's speed
// ratio, engine torque and losses at the crank speed) shared out over the lanes: one per lane of four,
// two per lane of two.  The maps lie in LDS, and a lane walks to the interval of this step's abscissa
// from the previous step's, which is nearly always the same one: an LDS read issued at the top of the step
// and two compares instead of a scan of every knot by scalar loads and a vector load of the segment found
// (for the HMMWV's four maps, 37 knots).  On ascending abscissae the walk ends at the interval the scan
// counts to (map_y), for any start.
constexpr int kGroupMaps = 4;
constexpr int kGroupMapEntries = kGroupMaps * kMaxMap;  // LDS entries of one wavefront

LFDM_HD const Map& group_map(const PSet& P, int id) {
    return id == kMapCf ? P.cfmap : id == kMapTr ? P.trmap : id == kMapTorque ? P.torque : P.losses;
}

// One lane's place on one map.
struct Walk {
    const MapXY* e;
    int r, n;  // interval (r - 1, r), entries
    MapXY first, last;
    double scale;  // factor on the ordinates
};

// tab: the wavefront's copies of the maps.
LFDM_HD void walk_init(const PSet& P, const MapXY* tab, double tqs, int id, Walk& w) {
    w.e = tab + id * kMaxMap;
    w.n = id == kMapCf ? P.cfmap.n : id == kMapTr ? P.trmap.n : id == kMapTorque ? P.torque.n : P.losses.n;
    w.r = 1;
    w.first = w.e[0];
    w.last = w.e[w.n > 0 ? w.n - 1 : 0];
    w.scale = id == kMapTorque ? tqs : 1.0;
}

// Walks to the interval of x; L, R: the segment of interval w.r, before and after.
LFDM_HD void walk_to(Walk& w, MapXY& L, MapXY& R, double x) {
    for (;;) {
        const bool down = w.r > 1 && !(L.x < x), up = w.r < w.n - 1 && R.x < x;
        if (!(down || up)) break;
        w.r += up ? 1 : -1;
        L = w.e[w.r - 1];
        R = w.e[w.r];
    }
}

// map_y (map_y_scaled with the ordinates' factor) at x; L, R: the segment of interval w.r.
LFDM_HD double walk(Walk& w, MapXY L, MapXY R, double x) {
    walk_to(w, L, R, x);
    const double ly = L.y * w.scale, ry = R.y * w.scale;
    const double mbar = fdiv(x - L.x, R.x - L.x);
    const double y = ly + mbar * (ry - ly);
    return x <= w.first.x ? w.first.y * w.scale : (x >= w.last.x ? w.last.y * w.scale : y);
}

// A lane's maps: its place's own of four, or two of them.
template <int G>
struct Walks {
    Walk a, b;  // b with two lanes only
};

template <int G>
LFDM_HD void walks_init(const PSet& P, const MapXY* tab, double tqs, int q, Walks<G>& w) {
    walk_init(P, tab, tqs, q, w.a);
    if (G == 2) walk_init(P, tab, tqs, 2 + q, w.b);
}

// The current gear's ratio, the ratio's reciprocal as fdiv refines it, and shift speeds; the places of a
// vehicle whose set the walk does not serve.
struct GearRow {
    double ratio, rcp, up, down;
    unsigned places = kNoPlaces;
};

LFDM_HD void gear_row(const PSet& P, int gear, GearRow& g) {
    const int i = gear_index(gear, P.ngears);
    g.ratio = P.gears[i];
    g.rcp = fdiv_rcp(g.ratio);
    g.up = P.shift[i].y;
    g.down = P.shift[i].x;
}

// Sets the walk does not serve (a map that does not ascend, or a torque map scaled by the throttle)
// scan their maps as the one-lane step does.
LFDM_HD bool group_walks(const PSet& P) {
    return !P.throttleMod && P.torque.sorted && P.losses.sorted && P.cfmap.sorted && P.trmap.sorted;
}

// The parameters a group step reads every step, held in the lane's registers.  A lone wavefront that fetches
// them through the scalar cache step by step waits for it some 28 times a step, a quarter of its time, and may
// use 512 registers: per step 2.69 -> 2.54 us (18-DOF, 16,384 vehicles, knots), 3.41 -> 3.24 (24-DOF), 2.62 ->
// 2.42 (11-DOF, 32,768).  Kernels of two wavefronts per SIMD, which hide each other's waits, have no room for
// them.  `full` has the maps and gears.
struct HotSet {
    double a, b, cf, cr, jxz, hrcf, hrcr, ks, bs, maxSteer;
    int nonLinearSteer, tcbool, driveType, whichWheels, ngears;
    TireP tire;
    Derived d;
    const PSet* full;
};

// Makes every double of t a register's value that the compiler cannot fetch again.
template <class T>
LFDM_HD void hold(T& t) {
    static_assert(sizeof(T) % sizeof(double) == 0, "doubles only");
    double* p = reinterpret_cast<double*>(&t);
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) / sizeof(double)); ++i) opaque(p[i]);
}

LFDM_HD void hot_init(const PSet& P, HotSet& h) {
    h.a = P.a; h.b = P.b; h.cf = P.cf; h.cr = P.cr; h.jxz = P.jxz; h.hrcf = P.hrcf; h.hrcr = P.hrcr;
    h.ks = P.ks; h.bs = P.bs; h.maxSteer = P.maxSteer;
    h.nonLinearSteer = P.nonLinearSteer; h.tcbool = P.tcbool; h.driveType = P.driveType;
    h.whichWheels = P.whichWheels; h.ngears = P.ngears;
    h.tire = P.tire;
    h.d = P.d;
    h.full = &P;
    for (double* v : {&h.a, &h.b, &h.cf, &h.cr, &h.jxz, &h.hrcf, &h.hrcr, &h.ks, &h.bs, &h.maxSteer}) opaque(*v);
    hold(h.tire);
    hold(h.d);
}

LFDM_HD const PSet& full_set(const PSet& P) { return P; }
LFDM_HD const PSet& full_set(const HotSet& h) { return *h.full; }

// The parameters a step reads: the set itself, or its HotSet in registers.
template <bool HOT>
struct Params {
    HotSet h;
    LFDM_HD void init(const PSet& P) { hot_init(P, h); }
    LFDM_HD const HotSet& of(const PSet&) const { return h; }
};
template <>
struct Params<false> {
    LFDM_HD void init(const PSet&) {}
    LFDM_HD const PSet& of(const PSet& P) const { return P; }
};

// powertrain_torque with the lookups and the gear's values of this vehicle's lanes.
template <int G, class PS>
LFDM_HD void powertrain_group(const PS& P, const Derived& u, double tqs, double throttle, double vel_u, double mean,
                              int q, bool walks, Walks<G>& w, GearRow& g, double& crank, int& gear,
                              double& torque_t, double& dcrank) {
    if (!walks) {
        powertrain_torque<false>(full_set(P), u, tqs, throttle, vel_u, mean, crank, gear, g.places, torque_t, dcrank);
        return;
    }
    const MapXY La = w.a.e[w.a.r - 1], Ra = w.a.e[w.a.r];
    MapXY Lb{}, Rb{};
    if constexpr (G == 2) {
        Lb = w.b.e[w.b.r - 1];
        Rb = w.b.e[w.b.r];
    }
    const double omega_out = fdiv_by(mean, g.ratio, g.rcp);
    double sr = 0;
    bool rev = false;
    if (P.tcbool) {
        const double quot = fdiv(omega_out, crank);
        sr = omega_out < 1e-9 || crank < 1e-9 ? 0.0 : quot;
        rev = sr > 1.;
        sr = rev ? 1. - (sr - 1.) : sr;
        sr = sr < 0 ? 0.0 : sr;
    } else {
        crank = omega_out;
    }
    double cf, tr, tq, loss;
    if constexpr (G == 4) {
        const double y = walk(w.a, La, Ra, q < 2 ? sr : crank);
        cf = group_value<4, kMapCf>(y);
        tr = group_value<4, kMapTr>(y);
        tq = group_value<4, kMapTorque>(y);
        loss = group_value<4, kMapLosses>(y);
    } else {
        const double ya = walk(w.a, La, Ra, sr), yb = walk(w.b, Lb, Rb, crank);
        cf = group_value<2, 0>(ya);
        tr = group_value<2, 1>(ya);
        tq = group_value<2, 0>(yb);
        loss = group_value<2, 1>(yb);
    }
    const double drive = tq * throttle + loss;
    if (P.tcbool) {
        const double c = fdiv(crank, cf);
        double torque_in = -(c * c);
        torque_in = rev ? -torque_in : torque_in;
        const double torque_out = rev ? -torque_in : -tr * torque_in;
        torque_t = fdiv_by(torque_out, g.ratio, g.rcp);
        dcrank = u.inv_ci * (drive + torque_in);
    } else {
        torque_t = fdiv_by(drive, g.ratio, g.rcp);
        dcrank = 0.0;
    }
    torque_t = vel_u < 1e-9 && torque_t < 0 ? 0.0 : torque_t;
    const int was = gear;
    if (omega_out > g.up) {
        if (gear < P.ngears - 1) gear++;
    } else if (omega_out < g.down) {
        if (gear > 0) gear--;
    }
    if (gear != was) gear_row(full_set(P), gear, g);
}

}  // namespace dev
}  // namespace lfdm
