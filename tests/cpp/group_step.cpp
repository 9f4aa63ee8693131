// Host build of the lane-group steps (csrc/d{11,18,24}_group.h) against the one-lane steps they must equal
// bit for bit.  A group's lanes run as threads that meet at every exchange (group.h's host_group_exchange),
// so the same code runs here as on the device, lane by lane.  Built by the Makefile's `groupstep`; loaded
// by tests/test_group_host.py.
#include <atomic>
#include <cstdio>
#include <string>
#include <thread>
#include <vector>

#include "../../low-fidelity-dynamic-models_amd/csrc/d18_group_adjoint.h"
#include "../../low-fidelity-dynamic-models_amd/csrc/integrate_group.h"
#include "../../low-fidelity-dynamic-models_amd/csrc/params.h"

using namespace lfdm;

namespace {

// The lanes of one group: every lane posts its value, waits for all, reads the one it wants, waits again.
struct Meeting {
    explicit Meeting(int n) : n(n) {}
    void meet() {
        const int turn = round.load(std::memory_order_acquire);
        if (arrived.fetch_add(1, std::memory_order_acq_rel) + 1 == n) {
            arrived.store(0, std::memory_order_relaxed);
            round.fetch_add(1, std::memory_order_acq_rel);
        } else {
            while (round.load(std::memory_order_acquire) == turn) std::this_thread::yield();
        }
    }
    double exchange(int lane, double v, int q) {
        post[lane] = v;
        meet();
        const double r = post[q];
        meet();
        return r;
    }
    const int n;
    double post[4];
    std::atomic<int> arrived{0}, round{0};
};

thread_local Meeting* t_meeting;
thread_local int t_lane;

double exchange(double v, int g, int q) {
    return t_meeting->exchange(t_lane, v, (t_lane & ~(g - 1)) + q);  // g 2 among four lanes: this lane's pair
}

struct Run {
    const PSet& P;
    const double* ovr;  // [7][n]
    const double* ctrl;  // [nsteps][3][n]
    int n, rec, nsteps;
    double dt;
};

kern::Ctl ctl(const Run& r, int i, int j) {
    const double* c = r.ctrl + (size_t)j * 3 * r.n + i;
    return {c[0], c[r.n], c[2 * r.n]};
}

// Both mirror the integration kernel's loop: every step but the last keeps the carried state and leaves its
// position update to the next, the last also returns the full record.
template <class M, bool NR>
void one_lane(const Run& r, double* st, int i) {
    typename M::S s;
    typename M::K k;
    typename M::X x;
    M::template load<NR>(st, r.n, i, s, k);
    M::kinit(r.P, r.ovr + i, r.n, k);
    for (int j = 0; j < r.nsteps; ++j) {
        if (j > 0) M::template position<false>(s, r.dt);
        if (j + 1 < r.nsteps)
            M::template step<NR, false, false, false>(r.P, r.P.d, k, s, ctl(r, i, j), r.dt, nullptr);
        else
            M::template step<NR, true, false, false>(r.P, r.P.d, k, s, ctl(r, i, j), r.dt, &x);
    }
    M::template position<false>(s, r.dt);
    M::template store<NR>(st, r.n, i, r.P, s, k, x);
}

template <class M, bool NR>
void group(const Run& r, double* st, int i) {
    std::vector<MapXY> tab(kGroupMapEntries);
    for (int id = 0; id < kGroupMaps; ++id)
        for (int e = 0; e < kMaxMap; ++e) tab[id * kMaxMap + e] = group_map(r.P, id).e[e];
    Meeting all(M::kLanes);
    std::vector<std::thread> lanes;
    for (int q = 0; q < M::kLanes; ++q)
        lanes.emplace_back([&, q] {
            t_meeting = &all;
            t_lane = q;
            host_group_exchange = exchange;
            typename M::S s;
            typename M::K k;
            typename M::X x;
            s.q = q;
            M::template load<NR>(st, r.n, i, s, k);
            M::kinit(r.P, r.ovr + i, r.n, tab.data(), s, k);
            for (int j = 0; j + 1 < r.nsteps; ++j)
                M::template step<NR, false>(r.P, r.P.d, k, s, ctl(r, i, j), r.dt, j > 0, nullptr);
            if (r.nsteps > 1) M::template position<false>(s, r.dt);
            M::template step<NR, true>(r.P, r.P.d, k, s, ctl(r, i, r.nsteps - 1), r.dt, false, &x);
            M::template position<false>(s, r.dt);
            all.meet();  // every lane has read the record before any writes it
            M::template store<NR>(st, r.n, i, r.P, s, k, x);
        });
    for (std::thread& t : lanes) t.join();
}

template <class M, bool NR, bool GROUP>
void run(const Run& r, const double* init, double* fin) {
    std::vector<double> st((size_t)r.rec * r.n);
    for (int i = 0; i < r.n; ++i)
        for (int f = 0; f < r.rec; ++f) st[(size_t)f * r.n + i] = init[(size_t)i * r.rec + f];
    for (int i = 0; i < r.n; ++i) {
        if constexpr (GROUP) group<M, NR>(r, st.data(), i);
        else one_lane<M, NR>(r, st.data(), i);
    }
    for (int i = 0; i < r.n; ++i)
        for (int f = 0; f < r.rec; ++f) fin[(size_t)i * r.rec + f] = st[(size_t)f * r.n + i];
}

template <class M, bool GROUP>
void pick_tire(const Run& r, int nr, const double* init, double* fin) {
    if (nr) run<M, true, GROUP>(r, init, fin);
    else run<M, false, GROUP>(r, init, fin);
}

}  // namespace

namespace {

// body(q, maps) on G lanes that exchange values.
template <int G, class F>
void on_lanes(const PSet& P, F body) {
    std::vector<MapXY> tab(kGroupMapEntries);
    for (int id = 0; id < kGroupMaps; ++id)
        for (int e = 0; e < kMaxMap; ++e) tab[id * kMaxMap + e] = group_map(P, id).e[e];
    Meeting all(G);
    std::vector<std::thread> lanes;
    for (int q = 0; q < G; ++q)
        lanes.emplace_back([&, q] {
            t_meeting = &all;
            t_lane = q;
            host_group_exchange = exchange;
            body(q, tab.data());
        });
    for (std::thread& t : lanes) t.join();
}

template <int G>
void adjoint_group(const PSet& P, AdjLaunch L, int nseg, int group) {
    for (int v = 0; v < L.n_user; ++v)
        on_lanes<G>(P, [&](int q, const MapXY* tab) { adj_forward_group<G, G == 4>(L, v, q, P, tab); });
    for (int hi = nseg; hi > 0; hi -= group) {
        L.seg_hi = hi;
        L.seg_lo = hi - group > 0 ? hi - group : 0;
        for (int v = 0; v < L.n_user; ++v) {
            if (hi < nseg)
                for (int q = 0; q < L.seg_hi - L.seg_lo; ++q) {
                    K18 k;
                    adj_recompute_lane(L, q, v, P, k);
                }
            // a lane's own storage here: the lanes write the same values, but are not in step
            on_lanes<G>(P, [&](int q, const MapXY* tab) {
                K18 k;
                K18b kb;
                adj_reverse_group<G>(L, v, q, P, tab, k, kb);
            });
        }
    }
}

// The reverse sweep over the whole tape with the kernel's own storage, shared as the kernel's lanes share it:
// the lanes here are not in step.
template <int G>
void adjoint_group_stored(const PSet& P, AdjLaunch L, int nseg) {
    for (int v = 0; v < L.n_user; ++v)
        on_lanes<G>(P, [&](int q, const MapXY* tab) { adj_forward_group<G, G == 4>(L, v, q, P, tab); });
    L.seg_hi = nseg;
    L.seg_lo = 0;
    for (int v = 0; v < L.n_user; ++v) {
        ReverseStore<G, G> store;
        on_lanes<G>(P, [&](int q, const MapXY* tab) {
            adj_reverse_group<G>(L, v, q, P, tab, store.constants(q), store.adjoints(q));
        });
    }
}

void adjoint_lanes(const PSet& P, AdjLaunch L, int nseg, int group) {
    for (int v = 0; v < L.n_user; ++v) adj_forward_lane(L, v, P);
    for (int hi = nseg; hi > 0; hi -= group) {
        L.seg_hi = hi;
        L.seg_lo = hi - group > 0 ? hi - group : 0;
        for (int v = 0; v < L.n_user; ++v) {
            K18 k;
            K18b kb;
            if (hi < nseg)
                for (int q = 0; q < L.seg_hi - L.seg_lo; ++q) adj_recompute_lane(L, q, v, P, k);
            adj_reverse_lane(L, v, P, k, kb);
        }
    }
}

}  // namespace

// Adjoint forward and backward of n <= 64 18-DOF vehicles on `lanes` lanes each, checkpoints every K steps and
// `group` segments per backward group: xy[nsteps][2][n], ctrl_bar[nsteps][3][n], state_bar[75][n],
// param_bar[7][n].  lanes -2 and -4: two and four, with the kernel's storage (group: all segments).
extern "C" int group_adjoint_run(int lanes, const double* flat, int len, const double* ovr, const double* init, int n,
                                 int nsteps, int K, int group, const double* ctrl, const double* xy_bar, double* xy,
                                 double* ctrl_bar, double* state_bar, double* param_bar) {
    PSet P;
    std::string e;
    if (n > 64 || !pset_from_flat(18, flat, len, 0, P, e)) return -1;
    const int S = 64, nseg = (nsteps + K - 1) / K;
    std::vector<double> st((size_t)75 * S, 0.0), ov((size_t)kOverrides * S, 1.0);
    std::vector<int> user(S, -1);
    for (int v = 0; v < n; ++v) {
        user[v] = v;
        for (int f = 0; f < 75; ++f) st[(size_t)f * S + v] = init[(size_t)v * 75 + f];
        for (int f = 0; f < kOverrides; ++f) ov[(size_t)f * S + v] = ovr[(size_t)f * n + v];
    }
    std::vector<double> ckpt((size_t)nseg * kAdjCkptRow * S), tape((size_t)group * K * kAdjTapeRow * S),
        carry((size_t)kAdjCarry * S);
    AdjLaunch L{};
    L.slot_user = user.data();
    L.state = st.data();
    L.ovr = ov.data();
    L.ctrl = ctrl;
    L.xy = xy;
    L.xy_bar = xy_bar;
    L.ctrl_bar = ctrl_bar;
    L.state_bar = state_bar;
    L.param_bar = param_bar;
    L.ckpt = ckpt.data();
    L.tape = tape.data();
    L.carry = carry.data();
    L.dt = 1e-3;
    L.nsteps = nsteps;
    L.K = K;
    L.S = S;
    L.n_user = n;
    L.fwd_tape_lo = nseg - group;
    if (lanes == 4) adjoint_group<4>(P, L, nseg, group);
    else if (lanes == 2) adjoint_group<2>(P, L, nseg, group);
    else if (lanes == -4) adjoint_group_stored<4>(P, L, nseg);
    else if (lanes == -2) adjoint_group_stored<2>(P, L, nseg);
    else adjoint_lanes(P, L, nseg, group);
    return 0;
}

// Step Jacobians jac[21][24][n] of n <= 64 vehicles at their records under ctrl[3][n]: by the kernel's rows, each
// through the parts of the step it reaches (full 0), or every row through the whole step (full 1).
extern "C" int group_jacobian_run(int full, const double* flat, int len, const double* ovr, const double* init, int n,
                                  const double* ctrl, double* jac) {
    PSet P;
    std::string e;
    if (n > 64 || !pset_from_flat(18, flat, len, 0, P, e)) return -1;
    const int S = 64;
    std::vector<double> st((size_t)75 * S, 0.0), ov((size_t)kOverrides * S, 1.0);
    std::vector<int> user(S, -1);
    for (int v = 0; v < n; ++v) {
        user[v] = v;
        for (int f = 0; f < 75; ++f) st[(size_t)f * S + v] = init[(size_t)v * 75 + f];
        for (int f = 0; f < kOverrides; ++f) ov[(size_t)f * S + v] = ovr[(size_t)f * n + v];
    }
    AdjLaunch L{};
    L.slot_user = user.data();
    L.state = st.data();
    L.ovr = ov.data();
    L.ctrl = ctrl;
    L.jac = jac;
    L.dt = 1e-3;
    L.S = S;
    L.n_user = n;
    for (int v = 0; v < n; ++v)
        for (int r = 0; r < kJacRows; ++r) {
            if (!full) {
                jac_row(L, r, v, P);
                continue;
            }
            S18 s;
            K18 k;
            load_record(L.state, S, v, s);
            load_k(P, L.ovr + v, S, k);
            S18b b;
            K18b kb;
            s18b_zero(b);
            k18b_zero(kb);
            double* seed[kJacRows] = {&b.xe[0], &b.ye[0], &b.xe[1], &b.ye[1], &b.xe[2], &b.ye[2], &b.xe[3],
                                      &b.ye[3], &b.omega[0], &b.omega[1], &b.omega[2], &b.omega[3], &b.crank, &b.x,
                                      &b.y, &b.u, &b.v, &b.psi, &b.wz, &b.phi, &b.wx};
            *seed[r] = 1.0;
            double g[3] = {0, 0, 0};
            step18_adj(P, P.d, k, s, ctrl[v], ctrl[n + v], ctrl[2 * n + v], L.dt, b, g[0], g[1], g[2], kb);
            double* row = jac + (size_t)r * kJacCols * n + v;
            for (int c = 0; c < kJacRows; ++c) row[(size_t)c * n] = c == 12 && !P.tcbool ? 0.0 : *seed[c];
            for (int c = 0; c < 3; ++c) row[(size_t)(kJacRows + c) * n] = g[c];
        }
    return 0;
}

// n vehicles, nsteps >= 1 steps on `lanes` lanes per vehicle (1, 2 or 4): final records into fin[n][rec].
// walks receives whether the group's map walk serves this parameter set.
extern "C" int group_step_run(int dof, int nr, int lanes, const double* flat, int len, const double* ovr,
                              const double* init, int n, int rec, int nsteps, const double* ctrl, double dt,
                              double* fin, int* walks) {
    PSet P;
    std::string e;
    if (!pset_from_flat(dof, flat, len, nr, P, e)) {
        std::fprintf(stderr, "%s\n", e.c_str());
        return -1;
    }
    *walks = group_walks(P) ? 1 : 0;
    const Run r{P, ovr, ctrl, n, rec, nsteps, dt};
    if (dof == 11 && lanes == 1) pick_tire<kern::M11, false>(r, nr, init, fin);
    else if (dof == 11 && lanes == 2) pick_tire<kern::M11g<true>, true>(r, nr, init, fin);
    else if (dof == 18 && lanes == 1) pick_tire<kern::M18, false>(r, nr, init, fin);
    else if (dof == 18 && lanes == 2) pick_tire<kern::M18g<2, false>, true>(r, nr, init, fin);
    else if (dof == 18 && lanes == 4) pick_tire<kern::M18g<4, true>, true>(r, nr, init, fin);
    else if (dof == 24 && lanes == 1) pick_tire<kern::M24, false>(r, nr, init, fin);
    else if (dof == 24 && lanes == 2) pick_tire<kern::M24g<2, false>, true>(r, nr, init, fin);
    else if (dof == 24 && lanes == 4) pick_tire<kern::M24g<4, true>, true>(r, nr, init, fin);
    else return -2;
    return 0;
}

// The driver table's lookups at nt times in turn, held rows (ahead) or not: steering, throttle, braking into
// out[nt][3].
extern "C" void driver_lookups(const double* rows, int n, const double* times, int nt, int ascending, int ahead,
                               double* out) {
    const DrvRow* r = reinterpret_cast<const DrvRow*>(rows);
    DrvWalk<false> w;
    DrvWalk<true> wa;
    for (int i = 0; i < nt; ++i, out += 3) {
        if (ahead) driver_input(times[i], r, n, ascending != 0, wa, out[0], out[1], out[2]);
        else driver_input(times[i], r, n, ascending != 0, w, out[0], out[1], out[2]);
    }
}

// Lookups on one map at nx abscissae in turn, each walking from the last one's place: the ordinates times sy.
extern "C" void map_lookups(const double* knots, int n, int sorted, const double* x, int nx, double sy, int id,
                            double* out) {
    Map m{};
    m.n = n;
    m.sorted = sorted;
    for (int i = 0; i < n; ++i) m.e[i] = {knots[2 * i], knots[2 * i + 1]};
    unsigned places = kNoPlaces;
    for (int i = 0; i < nx; ++i) out[i] = map_y_on<true>(m, find_segment(m, x[i], id, places), x[i], sy);
}

extern "C" int gear_row_of(int gear, int ngears) { return gear_index(gear, ngears); }

// The sine-step weights of pairs, together (out[4 i], out[4 i + 1]) and one by one (out[4 i + 2], out[4 i + 3]).
extern "C" void weight_pairs(const double* x, const double* y, int n, double* out) {
    for (int i = 0; i < n; ++i, out += 4) {
        sine_step_weights<false>(x[i], y[i], out[0], out[1]);
        out[2] = sine_step_weight<false>(x[i]);
        out[3] = sine_step_weight<false>(y[i]);
    }
}
