// Model traits of the lane-group steps (group.h) for the integration kernel: the records, launches and
// output rows of the one-lane traits in integrate.h, with each lane of a group loading and storing its own
// tires and lane 0 the chassis.
#pragma once
#include "d11_group.h"
#include "d18_group.h"
#include "d24_group.h"
#include "integrate.h"

namespace lfdm {
namespace kern {

// HOT: the set's parameters in registers (HotSet).
template <int G, bool HOT>
struct M18g {
    using S = S18g<G>;
    using X = X18g<G>;
    struct K {
        K18 c;
        K18g<G> g;
        Params<HOT> set;
    };
    static constexpr int kCh = M18::kCh;
    static constexpr bool kKInLds = false;  // a lane's registers hold its constants
    static constexpr int kLanes = G;
    static constexpr bool kAhead = HOT;
    static constexpr int N = S::N;
    template <bool NR>
    static LFDM_HD void load(const double* st, size_t S_, int slot, S& s, K&) {
        using Rr = M18::R<NR>;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const int i = N * s.q + j;
            if (!NR) {
                s.xe[j] = st[(size_t)(i * Rr::kTire + 0) * S_ + slot];
                s.ye[j] = st[(size_t)(i * Rr::kTire + 1) * S_ + slot];
                s.xedot[j] = st[(size_t)(i * Rr::kTire + 2) * S_ + slot];
                s.yedot[j] = st[(size_t)(i * Rr::kTire + 3) * S_ + slot];
            } else {
                s.xe[j] = s.ye[j] = s.xedot[j] = s.yedot[j] = 0.0;
            }
            s.omega[j] = st[(size_t)Rr::f(i, 0) * S_ + slot];
        }
        const double* v = st + (size_t)Rr::kVeh * S_ + slot;
        s.x = v[0 * S_]; s.y = v[1 * S_]; s.u = v[2 * S_]; s.v = v[3 * S_]; s.psi = v[4 * S_]; s.wz = v[5 * S_];
        s.phi = v[6 * S_]; s.wx = v[7 * S_]; s.udot = v[8 * S_]; s.vdot = v[9 * S_]; s.crank = v[12 * S_];
        s.gear = (int)v[14 * S_];
    }
    // o: the vehicle's parameters (stride S_), tab: the wavefront's maps
    static LFDM_HD void kinit(const PSet& P, const double* o, size_t S_, const MapXY* tab, S& s, K& k) {
        M18::kinit(P, o, S_, k.c);
        k18g_init<G>(P, k.c, s.q, k.g);
        k.set.init(P);
        walks_init<G>(P, tab, k.c.tqs, s.q, s.maps);
        gear_row(P, s.gear, s.row);
    }
    template <bool NR, bool FULL>
    static LFDM_HD void step(const PSet& P, const Derived&, const K& k, S& s, const Ctl& c, double dt, bool lag,
                             X* x) {
        const auto& h = k.set.of(P);
        double sd, cd;
        angles18g<G>(h, s, c.s, dt, lag, sd, cd);
        step18g<NR, FULL, G>(h, h.d, k.c, k.g, s, sd, cd, c.th, c.b, dt, x);
    }
    template <bool STRICT>
    static LFDM_HD void position(S& s, double dt) {
        double sp, cp;
        sincos_fast(s.psi, sp, cp);
        move18g<G>(s, sp, cp, dt);
    }
    static __device__ __forceinline__ void emit(double* o, size_t nu, double t, const S& s) {
#pragma unroll
        for (int j = 0; j < N; ++j) o[(size_t)(9 + N * s.q + j) * nu] = s.omega[j];
        if (s.q != 0) return;
        o[0 * nu] = t; o[1 * nu] = s.x; o[2 * nu] = s.y; o[3 * nu] = s.u; o[4 * nu] = s.v;
        o[5 * nu] = s.phi; o[6 * nu] = s.psi; o[7 * nu] = s.wx; o[8 * nu] = s.wz;
    }
    template <bool NR>
    static LFDM_HD void store(double* w, size_t S_, int slot, const PSet& P, const S& s, const K&, const X& x) {
        using Rr = M18::R<NR>;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const int i = N * s.q + j;
            if (!NR) {
                w[(size_t)(i * Rr::kTire + 0) * S_ + slot] = s.xe[j];
                w[(size_t)(i * Rr::kTire + 1) * S_ + slot] = s.ye[j];
                w[(size_t)(i * Rr::kTire + 2) * S_ + slot] = s.xedot[j];
                w[(size_t)(i * Rr::kTire + 3) * S_ + slot] = s.yedot[j];
            }
            const double f[11] = {s.omega[j], x.dOmega[j], x.xt[j], x.rStat[j], x.fx[j],    x.fy[j],
                                  x.fz[j],    x.vsx[j],    x.vsy[j], x.My[j],   x.engTor[j]};
#pragma unroll
            for (int m = 0; m < 11; ++m) w[(size_t)Rr::f(i, m) * S_ + slot] = f[m];
        }
        if (s.q != 0) return;
        double* v = w + (size_t)Rr::kVeh * S_ + slot;
        v[0 * S_] = s.x; v[1 * S_] = s.y; v[2 * S_] = s.u; v[3 * S_] = s.v; v[4 * S_] = s.psi; v[5 * S_] = s.wz;
        v[6 * S_] = s.phi; v[7 * S_] = s.wx; v[8 * S_] = s.udot; v[9 * S_] = s.vdot; v[10 * S_] = x.wxdot;
        v[11 * S_] = x.wzdot; v[12 * S_] = s.crank;
        if (P.tcbool) v[13 * S_] = x.dcrank;
        v[14 * S_] = (double)s.gear;
    }
};

template <bool HOT>
struct M11g {
    using S = S11g;
    using X = X11g;
    struct K {
        K11g g;
        Params<HOT> set;
    };
    static constexpr int kCh = M11::kCh;
    static constexpr bool kKInLds = false;
    static constexpr int kLanes = 2;
    static constexpr bool kAhead = HOT;
    template <bool NR>
    static LFDM_HD void load(const double* st, size_t S_, int slot, S& s, K&) {
        using Rr = M11::R<NR>;
        const int i = s.q;
        if (!NR) {
            s.xe = st[(size_t)(i * Rr::kTire + 0) * S_ + slot];
            s.ye = st[(size_t)(i * Rr::kTire + 1) * S_ + slot];
            s.xedot = st[(size_t)(i * Rr::kTire + 2) * S_ + slot];
            s.yedot = st[(size_t)(i * Rr::kTire + 3) * S_ + slot];
        } else {
            s.xe = s.ye = s.xedot = s.yedot = 0.0;
        }
        s.omega = st[(size_t)Rr::f(i, 0) * S_ + slot];
        const double* v = st + (size_t)Rr::kVeh * S_ + slot;
        s.x = v[0 * S_]; s.y = v[1 * S_]; s.u = v[2 * S_]; s.v = v[3 * S_]; s.psi = v[4 * S_]; s.wz = v[5 * S_];
        s.udot = v[6 * S_]; s.crank = v[9 * S_];
        s.gear = (int)v[11 * S_];
    }
    static LFDM_HD void kinit(const PSet& P, const double* o, size_t S_, const MapXY* tab, S& s, K& k) {
        K11 c;
        M11::kinit(P, o, S_, c);
        k11g_init(P, c, s.q, k.g);
        k.set.init(P);
        walks_init<2>(P, tab, c.tqs, s.q, s.maps);
        gear_row(P, s.gear, s.row);
    }
    template <bool NR, bool FULL>
    static LFDM_HD void step(const PSet& P, const Derived&, const K& k, S& s, const Ctl& c, double dt, bool lag,
                             X* x) {
        const auto& h = k.set.of(P);
        step11g<NR, FULL>(h, h.d, k.g, s, c.s, c.th, c.b, dt, lag, x);
    }
    template <bool STRICT>
    static LFDM_HD void position(S& s, double dt) {
        double sp, cp;
        sincos_fast(s.psi, sp, cp);
        move11g(s, sp, cp, dt);
    }
    static __device__ __forceinline__ void emit(double* o, size_t nu, double t, const S& s) {
        o[(size_t)(7 + s.q) * nu] = s.omega;
        if (s.q != 0) return;
        o[0 * nu] = t; o[1 * nu] = s.x; o[2 * nu] = s.y; o[3 * nu] = s.u; o[4 * nu] = s.v;
        o[5 * nu] = s.psi; o[6 * nu] = s.wz;
    }
    template <bool NR>
    static LFDM_HD void store(double* w, size_t S_, int slot, const PSet& P, const S& s, const K&, const X& x) {
        using Rr = M11::R<NR>;
        const int i = s.q;
        if (!NR) {
            w[(size_t)(i * Rr::kTire + 0) * S_ + slot] = s.xe;
            w[(size_t)(i * Rr::kTire + 1) * S_ + slot] = s.ye;
            w[(size_t)(i * Rr::kTire + 2) * S_ + slot] = s.xedot;
            w[(size_t)(i * Rr::kTire + 3) * S_ + slot] = s.yedot;
        }
        const double f[11] = {s.omega, x.dOmega, x.xt, x.rStat, x.fx, x.fy, x.fz, x.vsx, x.vsy, x.My, x.engTor};
#pragma unroll
        for (int m = 0; m < 11; ++m) w[(size_t)Rr::f(i, m) * S_ + slot] = f[m];
        if (s.q != 0) return;
        double* v = w + (size_t)Rr::kVeh * S_ + slot;
        v[0 * S_] = s.x; v[1 * S_] = s.y; v[2 * S_] = s.u; v[3 * S_] = s.v; v[4 * S_] = s.psi; v[5 * S_] = s.wz;
        v[6 * S_] = s.udot; v[7 * S_] = x.vdot; v[8 * S_] = x.wzdot; v[9 * S_] = s.crank;
        if (P.tcbool) v[10 * S_] = x.dcrank;
        v[11 * S_] = (double)s.gear;
    }
};

template <int G, bool HOT>
struct M24g {
    using S = S24g<G>;
    using X = X24g<G>;
    struct K {
        K24g<G> g;
        Params<HOT> set;
    };
    static constexpr int kCh = M24::kCh;
    static constexpr bool kKInLds = false;
    static constexpr int kLanes = G;
    static constexpr bool kAhead = HOT;
    static constexpr int N = S::N;
    template <bool NR>
    static LFDM_HD void load(const double* st, size_t S_, int slot, S& s, K& k) {
        using Rr = M24::R<NR>;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const int i = N * s.q + j;
            if (!NR) {
                s.xe[j] = st[(size_t)(i * Rr::kTire + 0) * S_ + slot];
                s.ye[j] = st[(size_t)(i * Rr::kTire + 1) * S_ + slot];
                s.xedot[j] = st[(size_t)(i * Rr::kTire + 2) * S_ + slot];
                s.yedot[j] = st[(size_t)(i * Rr::kTire + 3) * S_ + slot];
            } else {
                s.xe[j] = s.ye[j] = s.xedot[j] = s.yedot[j] = 0.0;
            }
            s.omega[j] = st[(size_t)Rr::f(i, 0) * S_ + slot];
            s.xt[j] = st[(size_t)Rr::f(i, 2) * S_ + slot];
            s.rStat[j] = st[(size_t)Rr::f(i, 4) * S_ + slot];
            k.g.vsz[j] = st[(size_t)Rr::f(i, 16) * S_ + slot];
            s.xs[j] = st[(size_t)Rr::q(i, 0) * S_ + slot];
            k.g.xsi[j] = st[(size_t)Rr::q(i, 1) * S_ + slot];
            s.dxs[j] = st[(size_t)Rr::q(i, 2) * S_ + slot];
            k.g.lsi[j] = st[(size_t)Rr::q(i, 4) * S_ + slot];
            s.wu[j] = st[(size_t)Rr::q(i, 13) * S_ + slot];
            s.fzd[j] = st[(size_t)Rr::q(i, 20) * S_ + slot];
        }
        const double* v = st + (size_t)Rr::kVeh * S_ + slot;
        s.x = v[0 * S_]; s.y = v[1 * S_]; s.u = v[3 * S_]; s.v = v[4 * S_]; s.w = v[5 * S_]; s.psi = v[6 * S_];
        s.wz = v[7 * S_]; s.phi = v[8 * S_]; s.wx = v[9 * S_]; s.theta = v[10 * S_]; s.wy = v[11 * S_];
        s.udot = v[12 * S_]; s.vdot = v[13 * S_]; s.wdot = v[14 * S_]; s.wxdot = v[15 * S_]; s.wydot = v[16 * S_];
        s.wzdot = v[17 * S_]; s.crank = v[21 * S_];
        s.gear = (int)v[23 * S_];
    }
    static LFDM_HD void kinit(const PSet& P, const double* o, size_t S_, const MapXY* tab, S& s, K& k) {
        K24 c;
        M24::kinit(P, o, S_, c);
        k24g_init<G>(P, c, s.q, k.g);
        k.set.init(P);
        walks_init<G>(P, tab, c.tqs, s.q, s.maps);
        gear_row(P, s.gear, s.row);
    }
    template <bool NR, bool FULL>
    static LFDM_HD void step(const PSet& P, const Derived&, const K& k, S& s, const Ctl& c, double dt, bool lag,
                             X* x) {
        const auto& h = k.set.of(P);
        step24g<NR, FULL, G>(h, h.d, k.g, s, c.s, c.th, c.b, dt, lag, x);
    }
    template <bool STRICT>
    static LFDM_HD void position(S& s, double dt) {
        double sp, cp;
        sincos_fast(s.psi, sp, cp);
        move24g<G>(s, sp, cp, dt);
    }
    static __device__ __forceinline__ void emit(double* o, size_t nu, double t, const S& s) {
#pragma unroll
        for (int j = 0; j < N; ++j) o[(size_t)(11 + N * s.q + j) * nu] = s.omega[j];
        if (s.q != 0) return;
        o[0 * nu] = t; o[1 * nu] = s.x; o[2 * nu] = s.y; o[3 * nu] = s.u; o[4 * nu] = s.v;
        o[5 * nu] = s.phi; o[6 * nu] = s.psi; o[7 * nu] = s.theta; o[8 * nu] = s.wx; o[9 * nu] = s.wz;
        o[10 * nu] = s.wy;
    }
    template <bool NR>
    static LFDM_HD void store(double* w, size_t S_, int slot, const PSet& P, const S& s, const K&, const X& x) {
        using Rr = M24::R<NR>;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const int i = N * s.q + j;
            if (!NR) {
                w[(size_t)(i * Rr::kTire + 0) * S_ + slot] = s.xe[j];
                w[(size_t)(i * Rr::kTire + 1) * S_ + slot] = s.ye[j];
                w[(size_t)(i * Rr::kTire + 2) * S_ + slot] = s.xedot[j];
                w[(size_t)(i * Rr::kTire + 3) * S_ + slot] = s.yedot[j];
            }
            // the fields and their order as in M24::store
            const double f[13] = {s.omega[j], x.dOmega[j], s.xt[j],   x.dxt[j],  s.rStat[j], x.fx[j], x.fy[j],
                                  x.fz[j],    x.fxg[j],    x.fyg[j],  x.fzg[j],  x.vgx[j],   x.vgy[j]};
#pragma unroll
            for (int m = 0; m < 13; ++m) w[(size_t)Rr::f(i, m) * S_ + slot] = f[m];
            w[(size_t)Rr::f(i, 14) * S_ + slot] = x.vsx[j];
            w[(size_t)Rr::f(i, 15) * S_ + slot] = x.vsy[j];
            w[(size_t)Rr::f(i, 17) * S_ + slot] = x.My[j];
            w[(size_t)Rr::f(i, 18) * S_ + slot] = x.engTor[j];
            w[(size_t)Rr::q(i, 0) * S_ + slot] = s.xs[j];
            w[(size_t)Rr::q(i, 2) * S_ + slot] = s.dxs[j];
            w[(size_t)Rr::q(i, 3) * S_ + slot] = x.ls[j];
            const double g[5] = {x.us[j], x.vs[j], x.ws[j], x.dus[j], x.dvs[j]};
#pragma unroll
            for (int m = 0; m < 5; ++m) w[(size_t)Rr::q(i, 5 + m) * S_ + slot] = g[m];
            const double h[13] = {x.uu[j],  x.vu[j],  s.wu[j],  x.duu[j], x.dvu[j], x.dwu[j], x.fxs[j],
                                  x.fys[j], x.fzs[j], s.fzd[j], x.mx[j],  x.my[j],  0.0};
#pragma unroll
            for (int m = 0; m < 13; ++m) w[(size_t)Rr::q(i, 11 + m) * S_ + slot] = h[m];
        }
        if (s.q != 0) return;
        double* v = w + (size_t)Rr::kVeh * S_ + slot;
        v[0 * S_] = s.x; v[1 * S_] = s.y; v[3 * S_] = s.u; v[4 * S_] = s.v; v[5 * S_] = s.w; v[6 * S_] = s.psi;
        v[7 * S_] = s.wz; v[8 * S_] = s.phi; v[9 * S_] = s.wx; v[10 * S_] = s.theta; v[11 * S_] = s.wy;
        v[12 * S_] = s.udot; v[13 * S_] = s.vdot; v[14 * S_] = s.wdot; v[15 * S_] = s.wxdot; v[16 * S_] = s.wydot;
        v[17 * S_] = s.wzdot; v[18 * S_] = x.dtheta; v[19 * S_] = x.dphi; v[20 * S_] = x.dpsi; v[21 * S_] = s.crank;
        if (P.tcbool) v[22 * S_] = x.dcrank;
        v[23 * S_] = (double)s.gear;
    }
};

}  // namespace kern
}  // namespace lfdm
