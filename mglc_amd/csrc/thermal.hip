// thermal.hip -- buoyancy-driven cavity on one MI355X: D3Q19 MRT flow with the
// Guo body force (Boussinesq + Coriolis) coupled to a D3Q7 MRT temperature
// field, fused into one pass per step or per two steps; the thermal residual and
// the Nusselt reductions.
//
// Reference step (bouyancy3d_mpi.F90:222-248, module.F90, evolution_f.F90,
// evolution_g.F90):
//   collision  (F from the previous rho, u, T; MRT + Guo source)
//   streaming, bounceback          (no-slip walls everywhere)
//   collisionT (previous u, T), streamingT, bouncebackT
//   macro (u = (sum f e + F/2) / rho), macroT (T = sum g)
// Stored between steps: f_post (19), g_post (7) and the force F of the last
// collision (macro of the next step needs F/2).  A step:
//   pull f and g (+ walls) -> macro with the stored F -> new F -> collide f
//   and g -> store.
// Device layout: the SoA layout of the isothermal path; g uses the same
// population stride; F is three arrays (only Fz is touched when the rotation rate
// is zero), of which a two-step launch reads one copy and writes another.
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>
#include <utility>

#include "collide.hpp"
#include "context.hpp"
#include "halo.hpp"
#include "plan.hpp"
#include "step.hpp"

using namespace lbm;

namespace {

struct ThermalArgs {
    const void* fsrc;
    void* fdst;
    const void* gsrc;
    void* gdst;
    void* force;  // Fx | Fy | Fz, each ps long (FP64 with FP64 storage, else FP32)
    int nx, ny, nz, px;
    long long pxy, ps;
    double snu, sq;           // flow rates (collision.f90:94-112 assignment)
    double para_a, qd, qnu;   // D3Q7: paraA, Qd = 3 - sqrt 3, Qnu = 4 sqrt 3 - 6
    double g_beta, omega_rot, t_ref;
    double t_hot, t_cold, cw; // held walls; cw = (6 + paraA) / 21
    int taxis;                // axis of the held walls (0 x, 1 y, 2 z), -1 none
    float scale, inv_scale;   // FP16 storage: populations held as value * 2^k
    unsigned seed;            // step number: drives the stochastic rounding of FP16 stores
    double *rho, *u, *v, *w, *T;
    // subdomain halo (the members the isothermal pull from outside reads):
    // faces in halo_faces take their incoming populations from `halo`
    int halo_faces;
    const void* halo;
    long long hoff[NREGION_ALL];
    double u_lid;             // 0: no moving lid here
};

// The stored body force: FP64 beside FP64 populations, else FP32 (the force
// is ~g beta ~ 1e-8, below FP16's normal range).
template <class S>
using ForceT = std::conditional_t<std::is_same_v<S, StoreF64>, double, float>;

// A stored population read by the buoyancy step: non-temporal in FP16
// storage.  Measured on MI355X at 128^3: FP16 62.9 -> 58.9 us per step;
// FP64 and FP32 ran no faster (171.8 and 82.5 us) and fetched 4 % more
// (lines shared by neighbouring blocks evicted sooner), and the cavity, batch
// and particle kernels ran 2-17 % slower, so those keep ordinary loads.
template <class S>
__device__ __forceinline__ typename S::Real ld_stream(const typename S::T* p) {
    if constexpr (S::BYTES == 2)
        return S::val(__builtin_nontemporal_load(p));
    else
        return ld<S>(p);
}

// Macro of the flow (evolution_f.F90:346-370) with the force F0 of the last
// collision (stored units): j holds J = sum e f + F0/2, u = J / rho.
template <class S, class R = typename S::Real>
__device__ __forceinline__ Moments<R> thermal_moments(const R f[Q], const R (&F0)[3], float inv_scale) {
#pragma clang fp contract(off)
    Moments<R> m;
    if constexpr (S::MOMENTS) population_sums_in_order(f, m.sum, m.j);
    else population_sums(f, m.sum, m.j);
    m.rho = density<S>(m.sum, inv_scale);
    for (int d = 0; d < 3; ++d) m.j[d] = fma_(R(0.5), F0[d], m.j[d]);
    if constexpr (S::MOMENTS) {
        velocity_by_division<S>(m, inv_scale);
    } else {
        const R r = rcp_near(m.rho);
        m.u = quotient(m.j[0], m.rho, r);
        m.v = quotient(m.j[1], m.rho, r);
        m.w = quotient(m.j[2], m.rho, r);
    }
    return m;
}

// A population of g bounced (bb) off a held wall (evolution_g.F90:60-197):
// -bb + (6 + paraA)/21 Twall, in stored units.
template <class S, class R = typename S::Real>
__device__ __forceinline__ R held_wall(const ThermalArgs& a, R bb, bool hot) {
#pragma clang fp contract(off)
    const R t = R(hot ? a.t_hot : a.t_cold);
    if constexpr (S::SCALED) return fma_(R(a.cw), t * R(a.scale), -bb);
    else return R(a.cw) * t - bb;
}

// The force of the next collision (evolution_f.F90:103-105) from this step's
// fields.
template <bool ROT, class R>
__device__ __forceinline__ void body_force(const ThermalArgs& a, const Moments<R>& q, R T, R (&F)[3]) {
#pragma clang fp contract(off)
    F[0] = ROT ? R(-2.0) * q.rho * q.v * R(a.omega_rot) : R(0.0);
    F[1] = ROT ? R(2.0) * q.rho * q.u * R(a.omega_rot) : R(0.0);
    F[2] = q.rho * R(a.g_beta) * (T - R(a.t_ref));
}

// The flow's collision with the new force F and the last one F0 (stored units).  In
// moments the force is formed here, its last products free to contract into the
// sums they go to.
template <class S, bool ROT, class R>
__device__ __forceinline__ void collide_flow_forced(const ThermalArgs& a, R (&f)[Q], const Moments<R>& q, R T,
                                                    const R (&F)[3], const R (&F0)[3]) {
    if constexpr (S::MOMENTS) {
        const R rho = S::SCALED ? q.rho * R(a.scale) : q.rho;
        const R Fc[3] = {ROT ? R(-2.0) * rho * q.v * R(a.omega_rot) : R(0.0),
                         ROT ? R(2.0) * rho * q.u * R(a.omega_rot) : R(0.0), rho * R(a.g_beta) * (T - R(a.t_ref))};
        collide_moments_forced<S>(f, q, Fc, R(a.snu), R(a.sq), a.scale);
    } else {
        collide_forced<S>(f, q, F, F0, R(a.snu), R(a.sq));
    }
}

// macroT (evolution_g.F90:202-218): T = sum g, in stored units.
template <class R>
__device__ __forceinline__ R temperature_sum(const R g[Q7]) {
    R T = g[0];
    sfor<Q7 - 1>([&](auto Am1) { T = T + g[decltype(Am1)::value + 1]; });
    return T;
}

// One step of the buoyancy-driven cavity.  S = StoreF64: FP64 arithmetic.
// StoreF32 / StoreF16: f stored as f - w (FP16
// scaled by 2^k with stochastic rounding), g stored unshifted (scaled the
// same way in FP16), the force in FP32, all arithmetic in FP32; the macro
// fields are written as FP64 for the FP64 reductions.
template <class S, bool ROT, bool MACRO, bool HALO>
__global__ __launch_bounds__(256) void k_thermal_step(const ThermalArgs a) {
    using ST = typename S::T;
    using R = typename S::Real;
    using FT = ForceT<S>;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    if (i >= a.nx || j >= a.ny) return;
    const int c = i + a.px * (j + a.ny * k);
    const ST* fsrc = static_cast<const ST*>(a.fsrc);
    const ST* gsrc = static_cast<const ST*>(a.gsrc);
    FT* force = static_cast<FT*>(a.force);

    // streaming + bounceback (evolution_f.F90:227-343): no-slip on all walls
    R f[Q];
    sfor<Q>([&](auto A) {
        constexpr int al = decltype(A)::value;
        constexpr int ex = EX[al], ey = EY[al], ez = EZ[al];
        if constexpr (al == 0) {
            f[0] = ld_stream<S>(fsrc + c);
        } else {
            bool in = true;
            if constexpr (ex != 0) in = in && (unsigned)(i - ex) < (unsigned)a.nx;
            if constexpr (ey != 0) in = in && (unsigned)(j - ey) < (unsigned)a.ny;
            if constexpr (ez != 0) in = in && (unsigned)(k - ez) < (unsigned)a.nz;
            const long long off = (long long)ex + (long long)ey * a.px + (long long)ez * a.pxy;
            if constexpr (HALO) {
                // from the halo where every crossed face borders a neighbour,
                // else bounce-back (no lid: top = false)
                f[al] = in ? ld_stream<S>(fsrc + (al * a.ps + c - off))
                           : pull_outside<S, COLL_MRT, al, true>(a, fsrc, i, j, k, c, false, 0.0);
            } else {
                f[al] = in ? ld_stream<S>(fsrc + (al * a.ps + c - off))
                           : ld_stream<S>(fsrc + (OPP[al] * a.ps + c));
            }
        }
    });
    // streamingT + bouncebackT (evolution_g.F90:60-197): adiabatic walls bounce
    // back; held walls: g(a) = -g_post(abar) + (6 + paraA)/21 Twall
    R g[Q7];
    sfor<Q7>([&](auto A) {
        constexpr int al = decltype(A)::value;
        constexpr int ex = EX[al], ey = EY[al], ez = EZ[al];
        if constexpr (al == 0) {
            g[0] = ld_stream<S>(gsrc + c);
        } else {
            constexpr int axis = ex != 0 ? 0 : (ey != 0 ? 1 : 2);
            constexpr int e = ex + ey + ez;
            const int q = axis == 0 ? i : (axis == 1 ? j : k);
            const int nq = axis == 0 ? a.nx : (axis == 1 ? a.ny : a.nz);
            const bool in = (unsigned)(q - e) < (unsigned)nq;
            const long long off = (long long)ex + (long long)ey * a.px + (long long)ez * a.pxy;
            constexpr int face = e > 0 ? 2 * axis : 2 * axis + 1;  // the face the pull enters through
            if (in) {
                g[al] = ld_stream<S>(gsrc + (al * a.ps + c - off));
            } else if (HALO && ((a.halo_faces >> face) & 1)) {
                // what arrives through `face`: the neighbour's D3Q7 population al
                const long long p = axis == 0 ? j + (long long)a.ny * k
                                              : (axis == 1 ? i + (long long)a.nx * k : i + (long long)a.nx * j);
                g[al] = ld_stream<S>(static_cast<const ST*>(a.halo) + (a.hoff[GREGION0 + face] + p));
            } else {
                const R bb = ld_stream<S>(gsrc + (OPP7[al] * a.ps + c));
                g[al] = (a.taxis == axis) ? held_wall<S>(a, bb, e > 0) : bb;
            }
        }
    });

    // macro (evolution_f.F90:346-370) with the force of the last collision
    const R unit = S::SCALED ? R(a.scale) : R(1);
    const R F0[3] = {ROT ? R(force[c]) * unit : R(0), ROT ? R(force[a.ps + c]) * unit : R(0),
                     R(force[2 * a.ps + c]) * unit};
    const Moments<R> q = thermal_moments<S>(f, F0, a.inv_scale);
    const R u = q.u, v = q.v, w = q.w;
    // macroT (evolution_g.F90:202-218)
    const R Ts = temperature_sum(g), T = S::SCALED ? Ts * R(a.inv_scale) : Ts;  // stored units, T
    if constexpr (MACRO) {
        const long long m = i + (long long)a.nx * (j + (long long)a.ny * k);
        a.rho[m] = density_f64<S>(q.sum, a.inv_scale);
        a.u[m] = double(u);
        a.v[m] = double(v);
        a.w[m] = double(w);
        a.T[m] = double(T);
    }
    R Fnew[3];  // next collision: force from this step's fields
    body_force<ROT>(a, q, T, Fnew);
    collide_flow_forced<S, ROT>(a, f, q, T, Fnew, F0);
    collide_d3q7<R>(g, Ts, u, v, w, R(a.para_a), R(a.qd), R(a.qnu));
    ST* fdst = static_cast<ST*>(a.fdst);
    ST* gdst = static_cast<ST*>(a.gdst);
    const unsigned h = cell_random<S>(c, a.seed);
    sfor<Q>([&](auto A) {
        constexpr int al = decltype(A)::value;
        st<S>(fdst + (al * a.ps + c), f[al], store_random<S, al>(h));
    });
    sfor<Q7>([&](auto A) {
        constexpr int al = decltype(A)::value;
        st<S>(gdst + (al * a.ps + c), g[al], store_random<S, Q + al>(h));
    });
    force[2 * a.ps + c] = FT(Fnew[2]);
    if constexpr (ROT) {
        force[c] = FT(Fnew[0]);
        force[a.ps + c] = FT(Fnew[1]);
    }
}

// ---- two steps in one pass ---------------------------------------------------------
// As pair.hpp does for the isothermal step (the tiles, the planes in LDS, the
// loads a plane ahead, the dropped stores): 26 populations per cell, so the LDS
// of a CU holds two planes of 384 cells in FP64 and 768 in FP32.  The force of
// the first step stays in the thread that made it; the one read and the one
// written lie in two arrays, since a rim cell's force is read by blocks that do
// not own it.  Same operations as k_thermal_step, same bits.
constexpr int QT = Q + Q7;

struct ThermalPairArgs : ThermalArgs {
    void* force_out;
    PairTiles t;
};

template <class S>
struct ThermalPairShape;
template <>
struct ThermalPairShape<StoreF64> {
    static constexpr int NT = 384, WAVES = 2;
};
template <>
struct ThermalPairShape<StoreF32> {
    static constexpr int NT = 768, WAVES = 3;
};

// Population n of a cell's 26: flow (0..18), then temperature, with its
// velocity and the opposite one's number.
constexpr int vel_of(int n) { return n < Q ? n : n - Q; }
constexpr int opp_of(int n) { return n < Q ? OPP[n] : Q + OPP7[n - Q]; }

template <class S, bool ROT, bool MACRO, bool EDGE, int NT>
__device__ __forceinline__ void thermal_pair(const ThermalPairArgs& a, int x0, int y0, int zs,
                                             typename S::T (&buf)[2][QT][NT]) {
    using T = typename S::T;
    using R = typename S::Real;
    using FT = ForceT<S>;
    const PairTiles& t = a.t;
    const int tid = threadIdx.x;
    const int cell = min(tid, t.w * t.h - 1);
    const int lx = cell % t.w, ly = cell / t.w;
    const int i = x0 + lx, j = y0 + ly;
    const bool own = tid < t.w * t.h && lx >= t.hx && lx < t.hx + t.tx && ly >= t.hy && ly < t.hy + t.ty &&
                     i < a.nx && j < a.ny;
    const int ci = min(max(i, 0), a.nx - 1), cj = min(max(j, 0), a.ny - 1);
    const int ze = min(zs + t.cz, a.nz);
    const int cxy = ci + a.px * cj;
    const int nbw = t.w;
    const int col = own || EDGE ? tid : nbw + 1;
    auto fresh = [](int v) {
        asm volatile("" : "+v"(v));
        return v;
    };
    // the pull of population n at plane k comes from inside the box (z: uniform)
    auto z_inside = [&](int ez, int k) { return ez == 0 || (ez > 0 ? k > 0 : k < a.nz - 1); };
    // population N of g, bounced (bb) off a wall that may be held at a temperature
    auto held = [&](auto N, R bb) {
        constexpr int v = vel_of(decltype(N)::value);
        constexpr int axis = EX[v] != 0 ? 0 : (EY[v] != 0 ? 1 : 2);
        return a.taxis == axis ? held_wall<S>(a, bb, EX[v] + EY[v] + EZ[v] > 0) : bb;
    };

    T in[QT];
    FT fin[3];  // the force of the last collision
    auto load = [&](int k) {
        const int cl = fresh(cxy);
        const long long plane = (long long)a.pxy * k;
        sfor<QT>([&](auto N) {
            constexpr int n = decltype(N)::value, v = vel_of(n);
            constexpr int ex = EX[v], ey = EY[v], ez = EZ[v];
            const T* s = static_cast<const T*>(n < Q ? a.fsrc : a.gsrc) + plane;
            constexpr int own_pop = n < Q ? n : n - Q, opp_pop = n < Q ? OPP[n < Q ? n : 0] : OPP7[n < Q ? 0 : n - Q];
            const bool zok = z_inside(ez, k);
            const long long from = (long long)own_pop * a.ps - (ex + (long long)ey * a.px + (long long)ez * a.pxy);
            const long long bounced = (long long)opp_pop * a.ps;
            if constexpr (EDGE && (ex != 0 || ey != 0)) {
                bool ok = zok;
                if constexpr (ex != 0) ok = ok && (unsigned)(ci - ex) < (unsigned)a.nx;
                if constexpr (ey != 0) ok = ok && (unsigned)(cj - ey) < (unsigned)a.ny;
                in[n] = s[cl + (ok ? from : bounced)];
            } else {
                in[n] = plane_load<T>(plane_of(s + (zok ? from : bounced)), (unsigned)cl * (unsigned)sizeof(T));
            }
        });
        const FT* fp = static_cast<const FT*>(a.force) + plane;
        for (int d = ROT ? 0 : 2; d < 3; ++d)
            fin[d] = plane_load<FT>(plane_of(fp + d * a.ps), (unsigned)cl * (unsigned)sizeof(FT));
    };
    // held walls: the pulls of g that came back from one (k: the plane)
    auto walls = [&](R(&g)[Q7], int k) {
        sfor<Q7 - 1>([&](auto Am1) {
            constexpr int n = Q + decltype(Am1)::value + 1, v = vel_of(n);
            std::integral_constant<int, n> N;
            if constexpr (EZ[v] != 0) {
                if (!z_inside(EZ[v], k)) g[v] = held(N, g[v]);
            } else if constexpr (EDGE) {
                const bool ok = EX[v] != 0 ? (unsigned)(ci - EX[v]) < (unsigned)a.nx
                                           : (unsigned)(cj - EY[v]) < (unsigned)a.ny;
                if (!ok) g[v] = held(N, g[v]);
            }
        });
    };
    // macro, force and collision of one cell (k_thermal_step's own): F0 the last
    // force, F the new one
    struct Fields {
        double rho;
        R u, v, w, T;
    };
    auto update = [&](R(&f)[Q], R(&g)[Q7], const R(&F0)[3], R(&F)[3]) {
        const Moments<R> q = thermal_moments<S>(f, F0, a.inv_scale);
        const R Ts = temperature_sum(g);
        body_force<ROT>(a, q, Ts, F);
        collide_flow_forced<S, ROT>(a, f, q, Ts, F, F0);
        collide_d3q7<R>(g, Ts, q.u, q.v, q.w, R(a.para_a), R(a.qd), R(a.qnu));
        return Fields{density_f64<S>(q.sum, a.inv_scale), q.u, q.v, q.w, Ts};
    };
    R made[3], before[3];  // the first step's force on the plane just made, and on the one below
    auto produce = [&](int p) {
        R f[Q], g[Q7], F0[3] = {R(0), R(0), R(0)};
        sfor<QT>([&](auto N) {
            constexpr int n = decltype(N)::value;
            if constexpr (n < Q) f[n] = S::val(in[n]);
            else g[n - Q] = S::val(in[n]);
        });
        for (int d = ROT ? 0 : 2; d < 3; ++d) F0[d] = R(fin[d]);
        walls(g, p);
        update(f, g, F0, made);
        sfor<QT>([&](auto N) {
            constexpr int n = decltype(N)::value;
            buf[p & 1][n][tid] = S::cvt(n < Q ? f[n < Q ? n : 0] : g[n < Q ? 0 : n - Q], 0u);
        });
    };
    auto pull = [&](auto N, int k, int c) {
        constexpr int n = decltype(N)::value, v = vel_of(n);
        constexpr int ex = EX[v], ey = EY[v], ez = EZ[v];
        const bool zok = z_inside(ez, k);
        const int plane = ez == 0 ? (k & 1) : ((k + 1) & 1);
        const int from = (plane * QT + n) * NT - (ex + ey * nbw), bounced = ((k & 1) * QT + opp_of(n)) * NT;
        const T* b = &buf[0][0][0];
        if constexpr (EDGE && (ex != 0 || ey != 0)) {
            bool ok = zok && own;
            if constexpr (ex != 0) ok = ok && (unsigned)(i - ex) < (unsigned)a.nx;
            if constexpr (ey != 0) ok = ok && (unsigned)(j - ey) < (unsigned)a.ny;
            return S::val(b[c + (ok ? from : bounced)]);
        } else {
            return S::val(b[c + (zok ? from : bounced)]);
        }
    };
    R up[6];  // the flow's five pulls along e_z = +1, and the temperature's
    auto take_up = [&](int k) {
        const int c = fresh(col);
        sfor<Q>([&](auto A) {
            constexpr int al = decltype(A)::value;
            if constexpr (EZ[al] > 0) up[up_slot(al)] = pull(A, k, c);
        });
        up[5] = pull(std::integral_constant<int, Q + 5>{}, k, c);
    };
    auto finish = [&](int k) {
        R f[Q], g[Q7], F[3] = {R(0), R(0), R(0)};
        const int c = fresh(col);
        sfor<QT>([&](auto N) {
            constexpr int n = decltype(N)::value, v = vel_of(n);
            if constexpr (n < Q) f[n] = EZ[v] > 0 ? up[EZ[v] > 0 ? up_slot(v) : 0] : pull(N, k, c);
            else g[n - Q] = EZ[v] > 0 ? up[5] : pull(N, k, c);
        });
        walls(g, k);
        const Fields m = update(f, g, before, F);
        if constexpr (MACRO) {
            if (own) {
                const long long mc = i + (long long)a.nx * (j + (long long)a.ny * k);
                a.rho[mc] = m.rho;
                a.u[mc] = double(m.u);
                a.v[mc] = double(m.v);
                a.w[mc] = double(m.w);
                a.T[mc] = double(m.T);
            }
        }
        const unsigned at = (unsigned)fresh(cxy);
        const long long plane = (long long)a.pxy * k;
        const unsigned where = own ? at * (unsigned)sizeof(T) : NOWHERE;
        sfor<QT>([&](auto N) {
            constexpr int n = decltype(N)::value;
            T* d = static_cast<T*>(n < Q ? a.fdst : a.gdst) + plane + (long long)vel_of(n) * a.ps;
            plane_store(S::cvt(n < Q ? f[n < Q ? n : 0] : g[n < Q ? 0 : n - Q], 0u), plane_of(d), where);
        });
        const unsigned fwhere = own ? at * (unsigned)sizeof(FT) : NOWHERE;
        FT* fp = static_cast<FT*>(a.force_out) + plane;
        for (int d = ROT ? 0 : 2; d < 3; ++d) plane_store(FT(F[d]), plane_of(fp + d * a.ps), fwhere);
    };

    const int p0 = max(zs - 1, 0), p1 = min(ze, a.nz - 1);
    made[0] = made[1] = made[2] = before[0] = before[1] = before[2] = R(0);
    load(p0);
    int p = p0;
    do {
        produce(p);
        load(min(p + 1, p1));
        lds_barrier();
        if (p == zs) take_up(p);
        // as many stores as the second step makes, all dropped
        sfor<QT>([&](auto N) {
            plane_store(T(0), plane_of(static_cast<T*>(a.fdst) + (long long)decltype(N)::value * 64), NOWHERE);
        });
        for (int d = ROT ? 0 : 2; d < 3; ++d)
            plane_store(FT(0), plane_of(static_cast<FT*>(a.force_out) + d * a.ps), NOWHERE);
        for (int d = 0; d < 3; ++d) before[d] = made[d];
        lds_barrier();
    } while (++p <= zs);
    for (; p <= p1; ++p) {
        produce(p);
        load(min(p + 1, p1));
        lds_barrier();
        finish(p - 1);
        for (int d = 0; d < 3; ++d) before[d] = made[d];
        take_up(p);
        lds_barrier();
    }
    if (ze == a.nz) finish(a.nz - 1);
}

template <class S, bool ROT, bool MACRO>
__global__ __launch_bounds__(ThermalPairShape<S>::NT, ThermalPairShape<S>::WAVES) void k_thermal_pair(
    const ThermalPairArgs a) {
    constexpr int NT = ThermalPairShape<S>::NT;
    __shared__ typename S::T buf[2][QT][NT];
    const int wg = xcd_order(blockIdx.x, gridDim.x);
    const PairTiles& t = a.t;
    const int bx = wg % t.ntx, by = (wg / t.ntx) % t.nty, bz = wg / (t.ntx * t.nty);
    const int x0 = bx * t.tx - t.hx, y0 = by * t.ty - t.hy;
    if (x0 >= 1 && x0 + t.w <= a.nx - 1 && y0 >= 1 && y0 + t.h <= a.ny - 1)
        thermal_pair<S, ROT, MACRO, false, NT>(a, x0, y0, bz * t.cz, buf);
    else
        thermal_pair<S, ROT, MACRO, true, NT>(a, x0, y0, bz * t.cz, buf);
}

// Equilibrium start (initial.F90:172-182) and the first collision from the
// given fields.  rho_in.. are compact nx*ny*nz arrays (also the macro output).
// The equilibria are formed in FP64 and the collision runs in the storage's
// arithmetic, as the step does.
template <class S, bool ROT>
__global__ __launch_bounds__(256) void k_thermal_init(const ThermalArgs a, const double* __restrict__ rho_in,
                                                      const double* __restrict__ u_in,
                                                      const double* __restrict__ v_in,
                                                      const double* __restrict__ w_in,
                                                      const double* __restrict__ T_in) {
    using R = typename S::Real;
    using FT = ForceT<S>;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    if (i >= a.nx || j >= a.ny) return;
    const int c = i + a.px * (j + a.ny * k);
    const long long m = i + (long long)a.nx * (j + (long long)a.ny * k);
    const double rho = rho_in[m], u = u_in[m], v = v_in[m], w = w_in[m], T = T_in[m];
    const double us2 = u * u + v * v + w * w;
    R f[Q], g[Q7];
    sfor<Q>([&](auto A) {
        constexpr int al = decltype(A)::value;
        const double un = u * EX[al] + v * EY[al] + w * EZ[al];
        const double feq = rho * weight(al) * (1.0 + 3.0 * un + 4.5 * un * un - 1.5 * us2);
        f[al] = S::SHIFT ? R((feq - weight(al)) * a.scale) : R(feq);
    });
    const double wt0 = (1.0 - a.para_a) / 7.0, wt1 = (a.para_a + 6.0) / 42.0;
    sfor<Q7>([&](auto A) {
        constexpr int al = decltype(A)::value;
        const double un = u * EX[al] + v * EY[al] + w * EZ[al];
        g[al] = R((al == 0 ? wt0 : wt1) * T * (1.0 + 21.0 / (6.0 + a.para_a) * un) * a.scale);
    });
    const double Fx = -2.0 * rho * v * a.omega_rot;
    const double Fy = 2.0 * rho * u * a.omega_rot;
    const double Fz = rho * a.g_beta * (T - a.t_ref);
    // f = f_eq carries the whole of rho u: no force before it (F0 = 0)
    const Moments<R> q = moments_of<S>(rho, u, v, w, a.scale);
    const R unit = S::SCALED ? R(a.scale) : R(1), F[3] = {R(Fx) * unit, R(Fy) * unit, R(Fz) * unit};
    const R F0[3] = {R(0), R(0), R(0)};
    if constexpr (S::MOMENTS) collide_moments_forced<S>(f, q, F, R(a.snu), R(a.sq), a.scale);
    else collide_forced<S>(f, q, F, F0, R(a.snu), R(a.sq));
    collide_d3q7<R>(g, R(T * a.scale), R(u), R(v), R(w), R(a.para_a), R(a.qd), R(a.qnu));
    using Tst = typename S::T;
    Tst* fdst = static_cast<Tst*>(a.fdst);
    Tst* gdst = static_cast<Tst*>(a.gdst);
    FT* force = static_cast<FT*>(a.force);
    const unsigned h = cell_random<S>(c, a.seed);
    sfor<Q>([&](auto A) {
        constexpr int al = decltype(A)::value;
        fdst[al * a.ps + c] = S::cvt(f[al], store_random<S, al>(h));
    });
    sfor<Q7>([&](auto A) {
        constexpr int al = decltype(A)::value;
        gdst[al * a.ps + c] = S::cvt(g[al], store_random<S, Q + al>(h));
    });
    force[c] = FT(Fx);
    force[a.ps + c] = FT(Fy);
    force[2 * a.ps + c] = FT(Fz);
    a.rho[m] = rho;
    a.u[m] = u;
    a.v[m] = v;
    a.w[m] = w;
    a.T[m] = T;
}

__device__ __forceinline__ double wave_sum(double x) {
    for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
    return x;
}

// Block-reduce NS sums into partial[NS * blockIdx.x + s].
template <int NS>
__device__ __forceinline__ void block_store(double (&e)[NS], double* partial) {
    __shared__ double sh[NS][RED_THREADS / 64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int s = 0; s < NS; ++s) {
        const double t = wave_sum(e[s]);
        if (lane == 0) sh[s][wid] = t;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        for (int s = 0; s < NS; ++s) {
            double t = 0.0;
            for (int q = 0; q < RED_THREADS / 64; ++q) t += sh[s][q];
            partial[NS * blockIdx.x + s] = t;
        }
}

// check.F90:16-41: e1 = sum |u - up|^2 (with w), e2 = sum |u|^2,
// e5 = sum |T - Tp|, e6 = sum |T|; then up = u, ..., Tp = T.
__global__ __launch_bounds__(RED_THREADS) void k_check_thermal(const double* __restrict__ u,
                                                               const double* __restrict__ v,
                                                               const double* __restrict__ w,
                                                               const double* __restrict__ T,
                                                               double* __restrict__ up, double* __restrict__ vp,
                                                               double* __restrict__ wp, double* __restrict__ Tp,
                                                               long long n, double* __restrict__ partial) {
    double e[4] = {0.0, 0.0, 0.0, 0.0};
    for (long long c = blockIdx.x * (long long)RED_THREADS + threadIdx.x; c < n;
         c += (long long)gridDim.x * RED_THREADS) {
        const double uu = u[c], vv = v[c], ww = w[c], tt = T[c];
        const double du = uu - up[c], dv = vv - vp[c], dw = ww - wp[c];
        e[0] += du * du + dv * dv + dw * dw;
        e[1] += uu * uu + vv * vv + ww * ww;
        e[2] += fabs(tt - Tp[c]);
        e[3] += fabs(tt);
        up[c] = uu;
        vp[c] = vv;
        wp[c] = ww;
        Tp[c] = tt;
    }
    block_store<4>(e, partial);
}

// Nusselt sums: s0 = sum w T over all cells (RaNu.F90:13-21), s1 = sum
// 2 (Thot - T) over the hot-wall layer (first layer along the held axis).
__global__ __launch_bounds__(RED_THREADS) void k_nusselt(const double* __restrict__ w,
                                                         const double* __restrict__ T, int nx, int ny, int nz,
                                                         int taxis, double t_hot, double* __restrict__ partial) {
    double e[2] = {0.0, 0.0};
    const long long n = (long long)nx * ny * nz;
    for (long long c = blockIdx.x * (long long)RED_THREADS + threadIdx.x; c < n;
         c += (long long)gridDim.x * RED_THREADS) {
        const double t = T[c];
        e[0] += w[c] * t;
        const long long i = c % nx, j = (c / nx) % ny, k = c / ((long long)nx * ny);
        const long long q = taxis == 0 ? i : (taxis == 1 ? j : k);
        if (q == 0) e[1] += (t_hot - t) * 2.0;
    }
    block_store<2>(e, partial);
}

template <int NS>
__global__ __launch_bounds__(RED_THREADS) void k_reduce_sums(const double* __restrict__ partial, int nblocks,
                                                             double* __restrict__ out) {
    double e[NS];
    for (int s = 0; s < NS; ++s) e[s] = 0.0;
    for (int b = threadIdx.x; b < nblocks; b += RED_THREADS)
        for (int s = 0; s < NS; ++s) e[s] += partial[NS * b + s];
    block_store<NS>(e, out);
}

ThermalArgs thermal_args(const lbm_ctx* c) {
    ThermalArgs a{};
    a.nx = c->p.nx;
    a.ny = c->p.ny;
    a.nz = c->p.nz;
    a.px = c->px;
    a.pxy = c->pxy;
    a.ps = c->ps;
    a.snu = 1.0 / c->p.tau;
    a.sq = 8.0 * (2.0 * c->p.tau - 1.0) / (8.0 * c->p.tau - 1.0);
    a.para_a = c->p.para_a;
    a.qd = 3.0 - std::sqrt(3.0);
    a.qnu = 4.0 * std::sqrt(3.0) - 6.0;
    a.g_beta = c->p.g_beta;
    a.omega_rot = c->p.omega_rot;
    a.t_ref = c->p.t_ref;
    a.t_hot = c->p.t_hot;
    a.t_cold = c->p.t_cold;
    a.cw = (6.0 + c->p.para_a) / 21.0;
    a.taxis = c->p.thermal_axis;
    a.scale = c->scale;
    a.inv_scale = c->inv_scale;
    a.force = c->force;
    a.rho = c->macro;
    a.u = c->macro + c->n;
    a.v = c->macro + 2 * c->n;
    a.w = c->macro + 3 * c->n;
    a.T = c->temp;
    a.halo_faces = c->p.halo_faces;
    a.halo = c->hin;
    for (int r = 0; r < NREGION_ALL; ++r) a.hoff[r] = c->hoff[r];
    a.u_lid = 0.0;
    return a;
}

dim3 thermal_grid(const lbm_ctx* c) {
    return dim3((c->p.nx + c->block.x - 1) / c->block.x, (c->p.ny + c->block.y - 1) / c->block.y,
                c->p.nz);
}

// Sum NS partial columns over RED_BLOCKS blocks into host `out`.
template <int NS>
int finish_sums(lbm_ctx* c, double* out) {
    hipLaunchKernelGGL(k_reduce_sums<NS>, dim3(1), dim3(RED_THREADS), 0, c->stream, c->red, RED_BLOCKS,
                       c->red + RED_MAX_SUMS * RED_BLOCKS);
    int rc = lbm_check_launch();
    if (rc) return rc;
    HIP_TRY(hipMemcpyAsync(out, c->red + RED_MAX_SUMS * RED_BLOCKS, NS * sizeof(double), hipMemcpyDeviceToHost,
                           c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return LBM_OK;
}

}  // namespace

size_t thermal_force_elem(const lbm_ctx* c) { return c->p.storage == LBM_STORE_F64 ? sizeof(double) : sizeof(float); }

// The tiles of the two-step kernel; false: one step per launch (FP16, which
// the rim's extra arithmetic slows; a loopback to rehearse; or where one-step launches are
// faster).
bool thermal_pair_plan(const lbm_params& p, int cus, PairTiles* t) {
    if (p.halo_loopback) return false;
    switch (p.storage) {
    case LBM_STORE_F64:
        // Up to 8 waves a CU the one-step kernel takes 8 to 11.8 us whatever the box (95 x
        // 66 x 15: 9.1, in pairs 11.0; 123 x 56 x 17 10.4 and 11.7; 64 x 67 x 26 10.2 and
        // 11.1; 57 x 35 x 57 11.7 both), past it 14 and more (62 x 55 x 42 15.7 and 13.0).
        return pair_plan(p.nx, p.ny, p.nz, ThermalPairShape<StoreF64>::NT, QT + 1, 8, {5.1, 1.2, 0.35, 8}, cus, t);
    case LBM_STORE_F32:
        return pair_plan(p.nx, p.ny, p.nz, ThermalPairShape<StoreF32>::NT, QT + 1, 4, {5.8, 1.3, 0.25}, cus, t);
    }
    return false;
}

int thermal_alloc(lbm_ctx* c) {
    const size_t g_bytes = (size_t)c->ps * Q7 * c->elem;
    const size_t f_bytes = 3 * (size_t)c->ps * thermal_force_elem(c);
    HIP_TRY(hipMalloc(&c->gbuf[0], g_bytes));
    HIP_TRY(hipMalloc(&c->gbuf[1], g_bytes));
    HIP_TRY(hipMalloc(&c->force_mem[0], f_bytes));
    c->force = c->force_mem[0];
    HIP_TRY(hipMalloc(&c->temp, (size_t)c->n * sizeof(double)));
    HIP_TRY(hipMalloc(&c->prev_t, 2 * (size_t)c->n * sizeof(double)));
    c->device_bytes += (long long)(2 * g_bytes + f_bytes + 3 * c->n * sizeof(double));
    return LBM_OK;
}

hipError_t thermal_alloc_next(lbm_ctx* c) {
    const int first = c->p.omega_rot != 0.0 ? 0 : 2;  // Fz alone without rotation
    const size_t component = (size_t)c->ps * thermal_force_elem(c), bytes = (3 - first) * component;
    const hipError_t e = hipMalloc(&c->force_mem[1], bytes);
    if (e != hipSuccess) return e;
    c->force_next = static_cast<char*>(c->force_mem[1]) - first * component;
    c->device_bytes += (long long)bytes;
    return e;
}

void thermal_release(lbm_ctx* c) {
    for (void* b : c->gbuf)
        if (b) (void)hipFree(b);
    for (void* m : c->force_mem)
        if (m) (void)hipFree(m);
    if (c->temp) (void)hipFree(c->temp);
    if (c->prev_t) (void)hipFree(c->prev_t);
}

namespace {

using ThermalFn = void (*)(const ThermalArgs);
using ThermalInitFn = void (*)(const ThermalArgs, const double*, const double*, const double*, const double*,
                               const double*);

template <class S>
struct ThermalTable {
    static constexpr ThermalFn step[2][2][2] = {
        {{k_thermal_step<S, false, false, false>, k_thermal_step<S, false, false, true>},
         {k_thermal_step<S, false, true, false>, k_thermal_step<S, false, true, true>}},
        {{k_thermal_step<S, true, false, false>, k_thermal_step<S, true, false, true>},
         {k_thermal_step<S, true, true, false>, k_thermal_step<S, true, true, true>}}};
    static constexpr ThermalInitFn init[2] = {k_thermal_init<S, false>, k_thermal_init<S, true>};
};

ThermalFn thermal_step_fn(const lbm_ctx* c, bool rot, bool macro, bool halo) {
    switch (c->p.storage) {
    case LBM_STORE_F32: return ThermalTable<StoreF32>::step[rot][macro][halo];
    case LBM_STORE_F16: return ThermalTable<StoreF16>::step[rot][macro][halo];
    default: return ThermalTable<StoreF64>::step[rot][macro][halo];
    }
}

using ThermalPairFn = void (*)(const ThermalPairArgs);

template <class S>
struct ThermalPairTable {
    // step[rotation][macro]
    static constexpr ThermalPairFn step[2][2] = {{k_thermal_pair<S, false, false>, k_thermal_pair<S, false, true>},
                                                 {k_thermal_pair<S, true, false>, k_thermal_pair<S, true, true>}};
};

int launch_thermal_pair(const lbm_ctx* c, const ThermalPairArgs& a, bool rot, bool macro) {
    const dim3 grid((unsigned)(a.t.ntx * a.t.nty * a.t.ncz));
    if (c->p.storage == LBM_STORE_F32)
        hipLaunchKernelGGL(ThermalPairTable<StoreF32>::step[rot][macro], grid, dim3(ThermalPairShape<StoreF32>::NT), 0,
                           c->stream, a);
    else
        hipLaunchKernelGGL(ThermalPairTable<StoreF64>::step[rot][macro], grid, dim3(ThermalPairShape<StoreF64>::NT), 0,
                           c->stream, a);
    return lbm_check_launch();
}

ThermalInitFn thermal_init_fn(const lbm_ctx* c, bool rot) {
    switch (c->p.storage) {
    case LBM_STORE_F32: return ThermalTable<StoreF32>::init[rot];
    case LBM_STORE_F16: return ThermalTable<StoreF16>::init[rot];
    default: return ThermalTable<StoreF64>::init[rot];
    }
}

}  // namespace

int thermal_load(lbm_ctx* c, const double* d_rho, const double* d_u, const double* d_v, const double* d_w,
                 const double* d_T) {
    ThermalArgs a = thermal_args(c);
    a.fdst = c->buf[0];
    a.gdst = c->gbuf[0];
    a.seed = (unsigned)c->itc;
    hipLaunchKernelGGL(thermal_init_fn(c, c->p.omega_rot != 0.0), thermal_grid(c), c->block, 0, c->stream, a, d_rho,
                       d_u, d_v, d_w, d_T);
    return lbm_check_launch();
}

// nsteps steps.  With halo_loopback the exchange runs before every step: the
// outgoing regions of the current state are packed and unpacked into the
// opposite faces' incoming regions (the regions the step reads).
int thermal_step(lbm_ctx* c, int nsteps) {
    ThermalArgs a = thermal_args(c);
    const bool rot = c->p.omega_rot != 0.0;
    const bool halo = c->p.halo_faces != 0;
    const bool loop = c->p.halo_loopback != 0;
    const dim3 grid = thermal_grid(c);
    ThermalPairArgs pa;
    pa.t = c->plan->pair;
    StepGroups groups(nsteps, c->plan->kind == StepPlan::PAIR && !step_capturing(c) ? 2 : 1);
    for (int s = 0; s < nsteps;) {
        if (loop) {
            int rc = halo_loopback_exchange(c);
            if (rc) return rc;
        }
        a.fsrc = c->buf[c->cur];
        a.fdst = c->buf[1 - c->cur];
        a.gsrc = c->gbuf[c->cur];
        a.gdst = c->gbuf[1 - c->cur];
        a.force = c->force;
        a.seed = (unsigned)(c->itc + s + 1);
        if (groups.next() == 2) {
            static_cast<ThermalArgs&>(pa) = a;
            pa.force_out = c->force_next;
            int rc = launch_thermal_pair(c, pa, rot, s + 2 == nsteps);
            if (rc) return rc;
            std::swap(c->force, c->force_next);
            s += 2;
        } else {
            hipLaunchKernelGGL(thermal_step_fn(c, rot, s == nsteps - 1, halo), grid, c->block, c->step_lds_halo,
                               c->stream, a);
            s += 1;
        }
        c->cur = 1 - c->cur;
    }
    return lbm_check_launch();
}

int thermal_check(lbm_ctx* c, double* sums4) {
    const long long n = c->n;
    hipLaunchKernelGGL(k_check_thermal, dim3(RED_BLOCKS), dim3(RED_THREADS), 0, c->stream, c->macro + n,
                       c->macro + 2 * n, c->macro + 3 * n, c->temp, c->prev, c->prev + n, c->prev_t,
                       c->prev_t + n, n, c->red);
    int rc = lbm_check_launch();
    if (rc) return rc;
    return finish_sums<4>(c, sums4);
}

// Sum of |u|^2 over all cells (calNuRe's Reynolds sum, RaNu.F90:36-44).
__global__ __launch_bounds__(RED_THREADS) void k_kinetic(const double* __restrict__ u, const double* __restrict__ v,
                                                         const double* __restrict__ w, long long n,
                                                         double* __restrict__ partial) {
    double e[1] = {0.0};
    for (long long c = blockIdx.x * (long long)RED_THREADS + threadIdx.x; c < n;
         c += (long long)gridDim.x * RED_THREADS)
        e[0] += u[c] * u[c] + v[c] * v[c] + w[c] * w[c];
    block_store<1>(e, partial);
}

int flow_reynolds(lbm_ctx* c, double* re) {
    hipLaunchKernelGGL(k_kinetic, dim3(RED_BLOCKS), dim3(RED_THREADS), 0, c->stream, c->macro + c->n,
                       c->macro + 2 * c->n, c->macro + 3 * c->n, c->n, c->red);
    int rc = lbm_check_launch();
    if (rc) return rc;
    double s[1];
    rc = finish_sums<1>(c, s);
    if (rc) return rc;
    const double viscosity = (c->p.tau - 0.5) / 3.0;
    *re = std::sqrt(s[0] / (double)c->n) * (double)c->p.nz / viscosity;
    return LBM_OK;
}

int thermal_nusselt(lbm_ctx* c, double* nu_vol, double* nu_wall) {
    const int ax = c->p.thermal_axis;
    if (ax < 0 || ax > 2) return lbm_fail(LBM_ERR_ARG, "lbm_nusselt: no held walls (thermal_axis = %d)", ax);
    const double* w = c->macro + 3 * c->n;  // gravity acts along z
    hipLaunchKernelGGL(k_nusselt, dim3(RED_BLOCKS), dim3(RED_THREADS), 0, c->stream, w, c->temp, c->p.nx, c->p.ny,
                       c->p.nz, ax, c->p.t_hot, c->red);
    int rc = lbm_check_launch();
    if (rc) return rc;
    double s[2];
    rc = finish_sums<2>(c, s);
    if (rc) return rc;
    const double kappa = (c->p.para_a + 6.0) / (42.0 * std::sqrt(3.0));  // inverse of module.F90:27
    const int na = ax == 0 ? c->p.nx : (ax == 1 ? c->p.ny : c->p.nz);
    const long long nwall = c->n / na;
    // calNuRe (RaNu.F90:21): <w T> nz / diffusivity + 1, whichever walls are held
    *nu_vol = s[0] / (double)c->n * (double)c->p.nz / kappa + 1.0;
    *nu_wall = s[1] / (double)nwall * (double)na / (c->p.t_hot - c->p.t_cold);
    return LBM_OK;
}
