// collide.hpp -- per-cell device arithmetic of the D3Q19 step: moments
// (macro), the collision (MRT, BGK, with and without a body force), the
// temperature's collision, and the population storage formats.  Everything
// here is unrolled at compile time over the lattice tables of lattice.hpp, so
// zero coefficients cost nothing and +-1 coefficients are plain adds.
//
// Two arithmetic spaces:
//   absolute  (SHIFT = false): registers hold f itself.  FP64 storage uses
//             this, so its operation order can follow the reference.
//   shifted   (SHIFT = true): registers hold g = f - w (the deviation from the
//             rest-state weights) and rho = 1 + drho.  FP32/FP16 storage use
//             it: deviations are O(Ma) small, so the 24-bit / 11-bit
//             mantissas are spent on the part that changes.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "lattice.hpp"

namespace lbm {

// ---- compile-time loop ------------------------------------------------------
template <class F, int... Is>
__device__ __forceinline__ void sfor_impl(F&& f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void sfor(F&& f) {
    sfor_impl(f, std::make_integer_sequence<int, N>{});
}

// acc + C*x with the multiply dropped for C = +-1.
template <int C, class R>
__device__ __forceinline__ R mac(R acc, R x) {
    if constexpr (C == 1) return acc + x;
    else if constexpr (C == -1) return acc - x;
    else return acc + R(C) * x;
}

// ---- storage formats ----------------------------------------------------------
// Registers hold populations in stored units: FP64 f itself, FP32 f - w, FP16
// (f - w) * 2^k as FP32.  The collision is linear in the populations apart from
// the velocity (a ratio) and rho = 1 + drho, so it runs in those units and only
// these two need the scale: no population is scaled on load or store, and a
// power-of-two scale changes no bit of the result.
// MOMENTS: the collision runs in the reference's 19 moments (collide_moments);
// else in pair form (relax).  FP16 keeps the moments: in pair form its kernel
// has 509 VALU instructions instead of 646 (256^3: 231 us a step against 241),
// but the last bits of a population then differ, and with them which way its
// store rounds, so that a run goes another, equally far off, way.
// Stores are non-temporal: the next step reads the written lattice only after
// the whole sweep, so caching the lines on the way out buys nothing (measured
// 2-4% faster at 256^3).
// Every cvt() and st() takes a 32-bit random word; only the FP16 format uses it.
struct StoreF64 {
    using T = double;
    using Real = double;
    static constexpr bool SHIFT = false;
    static constexpr bool SCALED = false;
    static constexpr bool MOMENTS = false;
    static constexpr bool RANDOM = false;
    static constexpr int BYTES = 8;
    __device__ __forceinline__ static Real val(T v) { return v; }
    __device__ __forceinline__ static T cvt(Real v, unsigned) { return v; }
};

struct StoreF32 {
    using T = float;
    using Real = float;
    static constexpr bool SHIFT = true;
    static constexpr bool SCALED = false;
    static constexpr bool MOMENTS = false;
    static constexpr bool RANDOM = false;
    static constexpr int BYTES = 4;
    __device__ __forceinline__ static Real val(T v) { return v; }
    __device__ __forceinline__ static T cvt(Real v, unsigned) { return v; }
};

// FP32 -> IEEE binary16 with stochastic rounding, on gfx950's conversion
// instruction (v_cvt_sr_f16_f32): the mantissa bits binary16 cannot hold are
// rounded up with probability equal to their value, driven by a uniform
// 32-bit word.  Rounding to nearest would round a slowly varying population
// the same way every step -- a constant spurious force that the flow
// integrates over its long viscous time; stochastic rounding makes that
// error unbiased.
__device__ __forceinline__ _Float16 to_half_stochastic(float x, unsigned rnd) {
    typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
    const half2_t h = __builtin_amdgcn_cvt_sr_f16_f32(half2_t{0, 0}, x, rnd, false);
    return h.x;
}

// Avalanche hash of a 32-bit word (the "lowbias32" integer mixer), used to
// draw the per-store random words from (cell, population, step).
__device__ __forceinline__ unsigned mix32(unsigned x) {
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}

// IEEE binary16 holding (f - w) * 2^k.  The scale is an exact power of two,
// so scaling adds no rounding; the store rounds stochastically.
struct StoreF16 {
    using T = _Float16;
    using Real = float;
    static constexpr bool SHIFT = true;
    static constexpr bool SCALED = true;
    static constexpr bool MOMENTS = true;
    static constexpr bool RANDOM = true;
    static constexpr int BYTES = 2;
    __device__ __forceinline__ static Real val(T v) { return static_cast<float>(v); }
    __device__ __forceinline__ static T cvt(Real v, unsigned rnd) { return to_half_stochastic(v, rnd); }
};

template <class S>
__device__ __forceinline__ typename S::Real ld(const typename S::T* p) {
    return S::val(*p);
}
template <class S>
__device__ __forceinline__ void st(typename S::T* p, typename S::Real v, unsigned rnd) {
    __builtin_nontemporal_store(S::cvt(v, rnd), p);
}

// Random words for the stores of cell c at step `seed`: one avalanche hash
// per cell, then a Weyl step per population.  Each word is uniform over cells
// and steps, which is what makes the rounding unbiased; one hash per cell
// keeps the store ALU-cheap.
template <class S>
__device__ __forceinline__ unsigned cell_random(long long c, unsigned seed) {
    if constexpr (S::RANDOM)
        return mix32((unsigned)c ^ (seed * 0x9E3779B9u));
    else
        return 0u;
}

template <class S, int a>
__device__ __forceinline__ unsigned store_random(unsigned h) {
    if constexpr (S::RANDOM)
        return h + (unsigned)a * 0x61C88647u;
    else
        return 0u;
}

enum { COLL_MRT = 0, COLL_BGK = 1 };

// The collision runs as the reference writes it (collide_moments), not in pair
// form.
template <class S, int COLL>
constexpr bool reference_form = S::MOMENTS || (COLL == COLL_BGK && sizeof(typename S::Real) == 8);

// ---- macroscopic moments (macro.f90:6-25) ---------------------------------------
template <class R>
struct Moments {
    R rho;       // density
    R sum;       // sum of the populations, in stored units: rho, or (rho - 1) * 2^k
    R j[3];      // sum of e_a f_a, in stored units
    R u, v, w;
};

__device__ __forceinline__ float rcp_near(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double rcp_near(double x) {
    const double r = __builtin_amdgcn_rcp(x);
    return __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
}
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }

// a / b given r = rcp_near(b), within a rounding or so of the exact quotient
// (the residual of the first product corrects it): three quotients by one rho
// cost one reciprocal and nine multiply-adds instead of three divisions.
template <class R>
__device__ __forceinline__ R quotient(R a, R b, R r) {
    const R q = a * r;
    return fma_(fma_(-q, b, a), r, q);
}

// rho, from the sum of the populations in stored units.
template <class S>
__device__ __forceinline__ typename S::Real density(typename S::Real sum, float inv_scale) {
    using R = typename S::Real;
    if constexpr (S::SCALED) return fma_(sum, inv_scale, R(1));
    else if constexpr (S::SHIFT) return R(1) + sum;
    else return sum;
}

// rho - 1 in stored units.
template <class S>
__device__ __forceinline__ typename S::Real excess(typename S::Real sum) {
    if constexpr (S::SHIFT) return sum;
    else return sum - 1.0;
}

// rho as the macro fields hold it.
template <class S>
__device__ __forceinline__ double density_f64(typename S::Real sum, float inv_scale) {
    if constexpr (S::SCALED) return 1.0 + double(sum * inv_scale);
    else if constexpr (S::SHIFT) return 1.0 + double(sum);
    else return sum;
}

// Sums of the populations and of e_a f_a from the sums and differences of
// opposite pairs, which the collision uses again (the compiler keeps one copy).
// No contraction here or in relax(): every kernel that updates a cell makes
// the same operations, so they agree bit for bit.
template <class R>
__device__ __forceinline__ void population_sums(const R f[Q], R& sum, R j[3]) {
#pragma clang fp contract(off)
    const R axis = ((f[1] + f[2]) + (f[3] + f[4])) + (f[5] + f[6]);
    const R diag = (((f[7] + f[10]) + (f[8] + f[9])) + ((f[11] + f[14]) + (f[12] + f[13]))) +
                   ((f[15] + f[18]) + (f[16] + f[17]));
    sum = (f[0] + axis) + diag;
    const R xy1 = f[7] - f[10], xy2 = f[8] - f[9];      // (1,1,0), (-1,1,0)
    const R xz1 = f[11] - f[14], xz2 = f[12] - f[13];   // (1,0,1), (-1,0,1)
    const R yz1 = f[15] - f[18], yz2 = f[16] - f[17];   // (0,1,1), (0,-1,1)
    j[0] = (f[1] - f[2]) + ((xy1 - xy2) + (xz1 - xz2));
    j[1] = (f[3] - f[4]) + ((xy1 + xy2) + (yz1 - yz2));
    j[2] = (f[5] - f[6]) + ((xz1 + xz2) + (yz1 + yz2));
}

// The same sums with a = 0..18 in order, as the reference accumulates them.
template <class R>
__device__ __forceinline__ void population_sums_in_order(const R f[Q], R& sum, R j[3]) {
    sum = f[0];
    for (int d = 0; d < 3; ++d) j[d] = R(-0.0);
    sfor<Q - 1>([&](auto B) {
        constexpr int a = decltype(B)::value + 1;
        sum = sum + f[a];
        if constexpr (EX[a] != 0) j[0] = mac<EX[a]>(j[0], f[a]);
        if constexpr (EY[a] != 0) j[1] = mac<EY[a]>(j[1], f[a]);
        if constexpr (EZ[a] != 0) j[2] = mac<EZ[a]>(j[2], f[a]);
    });
}

template <class S, class R = typename S::Real>
__device__ __forceinline__ void velocity_by_division(Moments<R>& m, float inv_scale) {
    if constexpr (S::SCALED) {
        m.u = m.j[0] * R(inv_scale) / m.rho;
        m.v = m.j[1] * R(inv_scale) / m.rho;
        m.w = m.j[2] * R(inv_scale) / m.rho;
    } else {
        m.u = m.j[0] / m.rho;
        m.v = m.j[1] / m.rho;
        m.w = m.j[2] / m.rho;
    }
}

template <class S, class R = typename S::Real>
__device__ __forceinline__ Moments<R> moments_in_order(const R f[Q], float inv_scale) {
    Moments<R> m;
    population_sums_in_order(f, m.sum, m.j);
    m.rho = density<S>(m.sum, inv_scale);
    velocity_by_division<S>(m, inv_scale);
    return m;
}

template <class S, int COLL, class R = typename S::Real>
__device__ __forceinline__ Moments<R> moments(const R f[Q], float inv_scale) {
#pragma clang fp contract(off)
    if constexpr (reference_form<S, COLL>) return moments_in_order<S>(f, inv_scale);
    Moments<R> m;
    population_sums(f, m.sum, m.j);
    m.rho = density<S>(m.sum, inv_scale);
    const R r = rcp_near(m.rho);
    m.u = quotient(m.j[0], m.rho, r);
    m.v = quotient(m.j[1], m.rho, r);
    m.w = quotient(m.j[2], m.rho, r);
    return m;
}

// Moments of a cell whose fields are given (the equilibrium starts).
template <class S, class R = typename S::Real>
__device__ __forceinline__ Moments<R> moments_of(double rho, double u, double v, double w, float scale) {
    Moments<R> m;
    m.rho = R(rho);
    m.sum = S::SHIFT ? R((rho - 1.0) * scale) : R(rho);
    m.j[0] = R(rho * u * scale);
    m.j[1] = R(rho * v * scale);
    m.j[2] = R(rho * w * scale);
    m.u = R(u);
    m.v = R(v);
    m.w = R(w);
    return m;
}

// ---- the collision (collision.f90:15-202, evolution_f.F90:58-129) --------------------
// The reference relaxes 19 moments m = M f.  Its rates are Snu on every even
// moment that is not conserved (e, eps, the stress rows 9..15), Sq on every odd
// one (q, m16..m18) and 0 on rho and j, and its equilibrium moments are those
// of the quadratic equilibrium f_eq (apart from row 12, below).  A space of
// moments that relaxes at one rate needs no basis: the even moments are the
// sums s = f_a + f_abar of opposite pairs (and f_0), the odd ones the
// differences d = f_a - f_abar (j, which must not change, is seen to below).
// So M, the rates and M^-1 are exactly
//   f_a, f_abar  +=  Snu/2 (s_eq - s)  +-  Sq/2 (d_eq - d).
// BGK is the case Sq = Snu = 1/tau.  Against the 19 x 19 transforms the FP32 step
// kernel went from 533 to 389 VALU instructions; FP64 and FP32, bound by memory,
// kept their time.
// The form updates f by the change alone, so a population's rounding error is
// that of the change and two sums instead of that of ten moments: after 300
// FP32 steps at 256^3 the velocity is 1e-7 off FP64 where it was 4e-6.  In
// FP64 (40 x 120 x 33, 400 steps, against 80-bit arithmetic) its rms error is
// 1.3e-16 where the transforms' is 2.5e-16.
// Mass and momentum are kept by construction, not by coefficients that cancel:
// f_0 loses what the pair sums gain, and the differences along the axes are
// what the diagonals leave of the momentum's gain.  Rounded weights
// (1/18, 1/36, 1/6) do not add up to 1, and in FP32 their few 1e-8 per step
// act on every cell the same way: mass drifted by 2.4e-7 in 20000 steps.
// FP64 follows the transforms in this: M^-1 in FP64 gives back 1 - 2^-54 of rho, so
// a run in transforms loses that share a step (measured over 20000 steps at 17^3,
// 64^3 and, with buoyancy, 128^3: 1.107e-12, 1.104e-12, 1.104e-12; the oracle at
// 128^3: 1.110e-12), and so does f_0 here (1.110e-12).  Without it the density is
// 1.1e-13 off a 64-bit run in transforms after 2000 steps at 17^3, with it 2e-15.
// BGK has no M^-1, and in FP64 is taken as the reference writes it.
//   base  Snu times the sum (rho or its excess), in stored units
//   C     Snu j: even part    w (base - 3/2 u.C + 9/2 (e.u)(e.C)) - Snu/2 s
//   B2    Sq j / 12: odd part of the diagonals   e.B2 - Sq/2 d
//   gain  half the momentum the collision adds (the body force), if any
//   k12   row 12's equilibrium of the cavity code lacks rho (collision.f90:85;
//         evolution_f.F90:75 has it): Snu (rho - 1)(v^2 - w^2) / 2 along row 12
//         of M^-1, which is -+1/12 on the y / z axes, +-1/24 on the xy / xz
//         diagonals
constexpr double TRANSFORM_LOSS = 0x1p-54;
template <bool ROW12, bool GAIN, class R>
__device__ __forceinline__ void relax(R f[Q], R sum, R base, const R (&C)[3], const R (&B2)[3], const R (&gain)[3], R u, R v,
                                      R w, R hs, R hd, R k12) {
#pragma clang fp contract(off)
    const R bb = fma_(R(-1.5), fma_(u, C[0], fma_(v, C[1], w * C[2])), base);
    R bax[3], bdi[3];  // the part common to a direction class: axes x, y, z; planes xy, xz, yz
    bax[0] = bax[1] = bax[2] = R(1.0 / 18.0) * bb;
    bdi[0] = bdi[1] = bdi[2] = R(1.0 / 36.0) * bb;
    if constexpr (ROW12) {
        bax[1] = fma_(R(-1.0 / 12.0), k12, bax[1]);
        bax[2] = fma_(R(1.0 / 12.0), k12, bax[2]);
        bdi[0] = fma_(R(1.0 / 24.0), k12, bdi[0]);
        bdi[1] = fma_(R(-1.0 / 24.0), k12, bdi[1]);
    }
    const R U[3] = {u, v, w};
    const R C1[3] = {R(0.25) * C[0], R(0.25) * C[1], R(0.25) * C[2]};
    const R C2[3] = {R(0.125) * C[0], R(0.125) * C[1], R(0.125) * C[2]};
    R x[NPAIR], y[NPAIR];  // what both members of a pair gain, and what the first gains over the second
    sfor<NPAIR>([&](auto P) {
        constexpr int p = decltype(P)::value, a = PAIR_A[p], b = OPP[a];
        constexpr int ex = EX[a], ey = EY[a], ez = EZ[a];
        const R s = f[a] + f[b];
        if constexpr (a < 7) {
            constexpr int d = ex ? 0 : (ey ? 1 : 2);
            x[p] = fma_(-hs, s, fma_(U[d], C1[d], bax[d]));
        } else {
            constexpr int d = ex ? 0 : 1, e = ez ? 2 : 1, pl = ez == 0 ? 0 : (ey == 0 ? 1 : 2);
            constexpr bool plus = (ex + ey + ez) == 2;  // else (-1 on d, +1 on e)
            const R eu = plus ? U[e] + U[d] : U[e] - U[d];
            const R ec = plus ? C2[e] + C2[d] : C2[e] - C2[d];
            const R eb = plus ? B2[e] + B2[d] : B2[e] - B2[d];
            x[p] = fma_(-hs, s, fma_(eu, ec, bdi[pl]));
            y[p] = fma_(-hd, f[a] - f[b], eb);
        }
    });
    // pairs 3..8: (1,1,0), (-1,1,0), (1,0,1), (-1,0,1), (0,1,1), (0,-1,1)
    static_assert(PAIR_A[3] == 7 && PAIR_A[4] == 8 && PAIR_A[5] == 11 && PAIR_A[6] == 12 && PAIR_A[7] == 15 &&
                  PAIR_A[8] == 16, "pair order");
    y[0] = (y[4] - y[3]) + (y[6] - y[5]);
    y[1] = (y[8] - y[7]) - (y[3] + y[4]);
    y[2] = -(y[5] + y[6]) - (y[7] + y[8]);
    if constexpr (GAIN)
        for (int d = 0; d < 3; ++d) y[d] = y[d] + gain[d];
    R even = (((x[0] + x[1]) + x[2]) + ((x[3] + x[4]) + (x[5] + x[6]))) + (x[7] + x[8]);
    if constexpr (sizeof(R) == 8) even = fma_(R(0.5 * TRANSFORM_LOSS), sum, even);
    f[0] = fma_(R(-2), even, f[0]);
    sfor<NPAIR>([&](auto P) {
        constexpr int p = decltype(P)::value, a = PAIR_A[p], b = OPP[a];
        f[a] = (f[a] + x[p]) + y[p];
        f[b] = (f[b] + x[p]) - y[p];
    });
}

// One isothermal collision with rates snu, sq (FP32 BGK: both 1/tau, no row 12).
template <class S, bool ROW12, class R = typename S::Real>
__device__ __forceinline__ void collide_flow(R f[Q], const Moments<R>& m, R snu, R sq, R row12) {
#pragma clang fp contract(off)
    const R b2 = R(1.0 / 12.0) * sq;
    const R C[3] = {snu * m.j[0], snu * m.j[1], snu * m.j[2]};
    const R B2[3] = {b2 * m.j[0], b2 * m.j[1], b2 * m.j[2]};
    R k12 = R(0);
    if constexpr (ROW12) k12 = (row12 * excess<S>(m.sum)) * fma_(m.v, m.v, -(m.w * m.w));
    relax<ROW12, false>(f, m.sum, snu * m.sum, C, B2, C, m.u, m.v, m.w, R(0.5) * snu, R(0.5) * sq, k12);
}

// The collision with the Guo source (evolution_f.F90:58-129): source moments
// scaled by 1 - s/2, momentum (rate 0) by 1, so it gains F.  m.j, m.u hold
// rho u = j + F0/2 with the force F0 of the last collision.  The source joins
// the equilibrium: C = Snu rho u + (2 - Snu) F, B = Sq rho u + (1 - Sq/2) F.
// The rate of the momentum rows of M^-1 (e / 10) is 0, not Sq: what Sq would
// take from them, Sq/2 (F - F0), is given back to every population.  Forces
// in stored units.
template <class S, class R = typename S::Real>
__device__ __forceinline__ void collide_forced(R f[Q], const Moments<R>& m, const R (&F)[3], const R (&F0)[3], R snu,
                                               R sq) {
#pragma clang fp contract(off)
    const R kc = R(2) - snu, kb = fma_(R(-0.5), sq, R(1)), kg = R(0.05) * sq;
    R C[3], B2[3], gain[3];
    for (int d = 0; d < 3; ++d) {
        C[d] = fma_(snu, m.j[d], kc * F[d]);
        B2[d] = fma_(R(1.0 / 12.0), fma_(sq, m.j[d], kb * F[d]), kg * (F[d] - F0[d]));
        gain[d] = R(0.5) * F[d];
    }
    relax<false, true>(f, m.sum, snu * m.sum, C, B2, gain, m.u, m.v, m.w, R(0.5) * snu, R(0.5) * sq, R(0));
}

// ---- moment transforms -----------------------------------------------------------------
// For the FP16 step, the fluid around spheres and the refill of uncovered nodes,
// which replaces moments.
// m = M f computed from the opposite-pair sums s_p = f_a + f_abar (even rows)
// and differences d_p = f_a - f_abar (odd rows); f_post = M^-1 m* likewise
// from even/odd partial sums E, O with f_a = E + O, f_abar = E - O.
template <class R>
__device__ __forceinline__ void mrt_forward(const R f[Q], R m[Q]) {
    R ps[NPAIR], pd[NPAIR];
    sfor<NPAIR>([&](auto P) {
        constexpr int p = decltype(P)::value;
        constexpr int a = PAIR_A[p];
        ps[p] = f[a] + f[OPP[a]];
        pd[p] = f[a] - f[OPP[a]];
    });
    sfor<Q>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr bool odd = row_is_odd(k);
        R acc = R(-0.0);
        if constexpr (!odd) acc = mac<basis(k, 0)>(acc, f[0]);
        sfor<NPAIR>([&](auto P) {
            constexpr int p = decltype(P)::value;
            constexpr int c = basis(k, PAIR_A[p]);
            if constexpr (c != 0) acc = mac<c>(acc, odd ? pd[p] : ps[p]);
        });
        m[k] = acc;
    });
}

template <class R>
__device__ __forceinline__ void mrt_inverse(const R m[Q], R f[Q]) {
    {
        R acc = R(-0.0);
        sfor<Q>([&](auto K) {
            constexpr int k = decltype(K)::value;
            constexpr int c = basis(k, 0);
            if constexpr (c != 0) acc = acc + R(double(c) / double(row_norm2(k))) * m[k];
        });
        f[0] = acc;
    }
    sfor<NPAIR>([&](auto P) {
        constexpr int a = PAIR_A[decltype(P)::value];
        R e = R(-0.0), o = R(-0.0);
        sfor<Q>([&](auto K) {
            constexpr int k = decltype(K)::value;
            constexpr int c = basis(k, a);
            if constexpr (c != 0) {
                constexpr R coef = R(double(c) / double(row_norm2(k)));
                if constexpr (row_is_odd(k)) o = o + coef * m[k];
                else e = e + coef * m[k];
            }
        });
        f[a] = e + o;
        f[OPP[a]] = e - o;
    });
}

// Equilibrium moments (collision.f90:73-91).  SHIFT: of rho = 1 + drho with M w =
// (1, -11, 3, 0, ...) subtracted, which leaves drho in rows 0..2.
// meq12_rho selects the thermal form -rho/2 (v^2 - w^2) (evolution_f.F90:75);
// the cavity form has no rho (collision.f90:85).  In stored units with rho, drho
// and one times the scale.
template <bool SHIFT, class R>
__device__ __forceinline__ void mrt_meq(R rho, R drho, R u, R v, R w, bool meq12_rho, R meq[Q], R one = R(1)) {
    const R us2 = u * u + v * v + w * w;
    if constexpr (SHIFT) {
        meq[0] = drho;
        meq[1] = R(-11) * drho + R(19) * rho * us2;
        meq[2] = R(3) * drho - R(11.0 / 2.0) * rho * us2;
    } else {
        meq[0] = rho;
        meq[1] = rho * (R(-11) + R(19) * us2);
        meq[2] = rho * (R(3) - R(11.0 / 2.0) * us2);
    }
    meq[3] = rho * u;
    meq[4] = R(-2.0 / 3.0) * rho * u;
    meq[5] = rho * v;
    meq[6] = R(-2.0 / 3.0) * rho * v;
    meq[7] = rho * w;
    meq[8] = R(-2.0 / 3.0) * rho * w;
    meq[9] = rho * (R(2) * u * u - v * v - w * w);
    meq[10] = R(-0.5) * rho * (R(2) * u * u - v * v - w * w);
    meq[11] = rho * (v * v - w * w);
    meq[12] = meq12_rho ? R(-0.5) * rho * (v * v - w * w) : R(-0.5) * one * (v * v - w * w);
    meq[13] = rho * u * v;
    meq[14] = rho * v * w;
    meq[15] = rho * u * w;
    meq[16] = R(0);
    meq[17] = R(0);
    meq[18] = R(0);
}

// Rates (collision.f90:94-112): 0 on rho and j, Snu = 1/tau on e, eps and the
// stress rows 9..15, Sq = 8(2tau-1)/(8tau-1) on q and m16..18.
template <int k>
constexpr int rate_kind() {
    return (k == 0 || k == 3 || k == 5 || k == 7) ? 0 : ((k == 4 || k == 6 || k == 8 || k >= 16) ? 2 : 1);
}

// The collision in the moments' own form (collision.f90:15-202; BGK:
// collision.f90:192-198, feq of initial.f90:63-73), for moments_in_order.  With
// f - w stored the w-part of feq drops out: w (drho + rho (3 e.u + 4.5 (e.u)^2 -
// 1.5 u.u)).
template <class S, bool BGK, class R = typename S::Real>
__device__ __forceinline__ void collide_moments(R f[Q], const Moments<R>& q, R snu, R sq, bool meq12_rho, float scale) {
    R one = R(1), rho = q.rho;
    if constexpr (S::SCALED) {
        one = R(scale);
        rho = q.rho * one;
    }
    if constexpr (BGK) {
        const R us2 = q.u * q.u + q.v * q.v + q.w * q.w;
        // FP64: contracted by hand, the same in every kernel (left to the compiler the
        // block kernel's came out otherwise)
        const R us2c = fma_(q.w, q.w, fma_(q.u, q.u, q.v * q.v));
        sfor<Q>([&](auto B) {
            constexpr int a = decltype(B)::value;
            R un = R(-0.0);
            if constexpr (EX[a] != 0) un = mac<EX[a]>(un, q.u);
            if constexpr (EY[a] != 0) un = mac<EY[a]>(un, q.v);
            if constexpr (EZ[a] != 0) un = mac<EZ[a]>(un, q.w);
            constexpr R wa = R(weight(a));
            if constexpr (S::SHIFT) {
                const R feq = wa * (q.sum + rho * (R(3) * un + R(4.5) * un * un - R(1.5) * us2));
                f[a] = f[a] - snu * (f[a] - feq);
            } else {
                const R X = fma_(R(-1.5), us2c, fma_(R(4.5) * un, un, fma_(R(3), un, R(1))));
                f[a] = fma_(-snu, fma_(-(rho * wa), X, f[a]), f[a]);
            }
        });
    } else {
        R m[Q], meq[Q];
        mrt_forward(f, m);
        mrt_meq<S::SHIFT>(rho, q.sum, q.u, q.v, q.w, meq12_rho, meq, one);
        sfor<Q>([&](auto K) {
            constexpr int k = decltype(K)::value;
            constexpr int kind = rate_kind<k>();
            if constexpr (kind == 1) m[k] = m[k] - snu * (m[k] - meq[k]);
            else if constexpr (kind == 2) m[k] = m[k] - sq * (m[k] - meq[k]);
        });
        mrt_inverse(m, f);
    }
}

// The same with the Guo source in moment space (evolution_f.F90:58-129):
// m* = m - s (m - meq) + (1 - s/2) S, meq in the thermal form (row 12 with rho).
// Forces in stored units.
template <class S, class R = typename S::Real>
__device__ __forceinline__ void collide_moments_forced(R f[Q], const Moments<R>& q, const R (&F)[3], R snu, R sq,
                                                       float scale) {
    const R u = q.u, v = q.v, w = q.w, rho = S::SCALED ? q.rho * R(scale) : q.rho;
    const R Fx = F[0], Fy = F[1], Fz = F[2];
    R m[Q], meq[Q], s[Q];
    mrt_forward(f, m);
    const R us2 = u * u + v * v + w * w;
    meq[0] = q.sum;
    meq[1] = R(-11.0) * q.sum + R(19.0) * rho * us2;
    meq[2] = R(3.0) * q.sum - R(11.0 / 2.0) * rho * us2;
    meq[3] = rho * u;
    meq[4] = R(-2.0 / 3.0) * meq[3];
    meq[5] = rho * v;
    meq[6] = R(-2.0 / 3.0) * meq[5];
    meq[7] = rho * w;
    meq[8] = R(-2.0 / 3.0) * meq[7];
    meq[9] = rho * (R(2.0) * u * u - v * v - w * w);
    meq[10] = R(-0.5) * meq[9];
    meq[11] = rho * (v * v - w * w);
    meq[12] = R(-0.5) * meq[11];
    meq[13] = rho * (u * v);
    meq[14] = rho * (v * w);
    meq[15] = rho * (w * u);
    meq[16] = meq[17] = meq[18] = R(0.0);
    const R uF = u * Fx + v * Fy + w * Fz;
    s[0] = R(0.0);
    s[1] = R(38.0) * uF;
    s[2] = R(-11.0) * uF;
    s[3] = Fx;
    s[4] = R(-2.0 / 3.0) * Fx;
    s[5] = Fy;
    s[6] = R(-2.0 / 3.0) * Fy;
    s[7] = Fz;
    s[8] = R(-2.0 / 3.0) * Fz;
    s[9] = R(4.0) * u * Fx - R(2.0) * v * Fy - R(2.0) * w * Fz;
    s[10] = R(-2.0) * u * Fx + v * Fy + w * Fz;
    s[11] = R(2.0) * v * Fy - R(2.0) * w * Fz;
    s[12] = -v * Fy + w * Fz;
    s[13] = u * Fy + v * Fx;
    s[14] = v * Fz + w * Fy;
    s[15] = u * Fz + w * Fx;
    s[16] = s[17] = s[18] = R(0.0);
    sfor<Q>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int kind = rate_kind<k>();
        if constexpr (kind == 0) m[k] = m[k] + s[k];
        else if constexpr (kind == 1) m[k] = m[k] - snu * (m[k] - meq[k]) + (R(1.0) - R(0.5) * snu) * s[k];
        else m[k] = m[k] - sq * (m[k] - meq[k]) + (R(1.0) - R(0.5) * sq) * s[k];
    });
    mrt_inverse(m, f);
}

// D3Q7 MRT for the temperature (evolution_g.F90:1-57): n = N g,
// neq = (T, T u, T v, T w, T paraA, 0, 0), rates (0, Qd x3, Qnu x3),
// g_post = N^-1 n*, N^-1 = N^T diag(1/|row|^2).  g is stored unshifted; T
// in g's units.  (In pair form, as the flow, this would keep T in FP32 where the
// rounded 1/7, 1/42, ... move it by 4e-8 per step, 2.8e-5 of the change of T
// over 120 steps at 128^3; the transforms stay so that FP32 fields do not move by
// more than their own rounding from one version to the next.)
template <class R>
__device__ __forceinline__ void collide_d3q7(R g[Q7], R T, R u, R v, R w, R para_a, R qd, R qnu) {
    R n[Q7];
    sfor<Q7>([&](auto K) {
        constexpr int k = decltype(K)::value;
        R acc = R(-0.0);
        sfor<Q7>([&](auto A) {
            constexpr int a = decltype(A)::value;
            constexpr int c = basis7(k, a);
            if constexpr (c != 0) acc = mac<c>(acc, g[a]);
        });
        n[k] = acc;
    });
    const R neq[Q7] = {T, T * u, T * v, T * w, T * para_a, R(0.0), R(0.0)};
    sfor<Q7>([&](auto K) {
        constexpr int k = decltype(K)::value;
        if constexpr (k >= 1 && k <= 3) n[k] = n[k] - qd * (n[k] - neq[k]);
        else if constexpr (k >= 4) n[k] = n[k] - qnu * (n[k] - neq[k]);
    });
    sfor<Q7>([&](auto A) {
        constexpr int a = decltype(A)::value;
        R acc = R(-0.0);
        sfor<Q7>([&](auto K) {
            constexpr int k = decltype(K)::value;
            constexpr int c = basis7(k, a);
            if constexpr (c != 0) acc = acc + R(double(c) / double(row_norm2_7(k))) * n[k];
        });
        g[a] = acc;
    });
}

}  // namespace lbm
