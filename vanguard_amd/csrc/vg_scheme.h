// The SLIC / FORCE building blocks, generic over the physics P (Euler, MHD,
// HPR) and the sweep direction, on register arrays.  EXACT mode follows the
// reference's operation order (see the citations) with every product and sum
// rounded separately; FAST mode is the same scheme with the primitive/conserved
// round trips removed and multiply-adds fused (fp contract(on) in its branches
// only: a product is fused into the sum of its own expression, so every kernel
// that inlines this code rounds alike, whatever its shape).
#pragma once

#include "vg_device.h"
#include "vg_quot.h"

namespace vg {

enum { MODE_EXACT = 0, MODE_FAST = 1 };

// Physics whose EXACT conversions can hand the shared divisor of rho from a
// primitive conversion to the flux of the same density (cons_to_prim_d, flux_d).
template <class P, class = void>
struct HasSharedDivisor {
    static constexpr bool value = false;
};
template <class P>
struct HasSharedDivisor<P, decltype((void)&P::template flux_d<0>)> {
    static constexpr bool value = true;
};

// Physics whose conversion to primitives, back, and flux share one divisor in a
// function of their own (round_trip), a side at a time: two sides of the 17-field
// state side by side would not fit the registers.
template <class P, class = void>
struct HasRoundTrip {
    static constexpr bool value = false;
};
template <class P>
struct HasRoundTrip<P, decltype((void)&P::template round_trip<0>)> {
    static constexpr bool value = true;
};

// Physics whose FAST flux comes less another flux in the same expressions
// (flux_less_fast), its products fused into the differences, as they are not across
// statements (4096 x 4096, 4 fields: x walk 257 us a sweep without, 247 so).
template <class P, class = void>
struct HasFluxLess {
    static constexpr bool value = false;
};
template <class P>
struct HasFluxLess<P, decltype((void)&P::template flux_less_fast<0>)> {
    static constexpr bool value = true;
};

// Correctly rounded division: the compiler's IEEE division, or the division
// sequence without its scaling steps where the caller has shown the operands
// in range (vg_quot.h).
struct IeeeDiv {
    __device__ __forceinline__ double operator()(double a, double b) const { return a / b; }
};
struct InRangeDiv {
    __device__ __forceinline__ double operator()(double a, double b) const { return div_in_range(a, b); }
};

// SlopeLimiters::computeRCoefficient and computeSlopeLimiter
// (Solvers/slopelimiters.cpp:7-74): 0 superbee, 1 van Leer, anything else minbee.
template <class Div = IeeeDiv>
__device__ __forceinline__ double r_coefficient(double r, double bias, Div div = Div())
{
    return div(2.0, (1.0 - bias) + ((1.0 + bias) * r));
}

template <class Div = IeeeDiv>
__device__ __forceinline__ double limiter_value(double r, double bias, int limiter, Div div = Div())
{
    if (r < 0.0) return 0.0;
    if (limiter == 0) {
        if (r < 0.5) return 2.0 * r;
        if (r < 1.0) return 1.0;
        return smin(smin(r, r_coefficient(r, bias, div)), 2.0);
    }
    if (limiter == 1) return smin(div(2.0 * r, 1.0 + r), r_coefficient(r, bias, div));
    if (r < 1.0) return r;
    return smin(1.0, r_coefficient(r, bias, div));
}

// The limiter's divisions are in the range of the short division sequence when
// every slope difference is at most 2^600 in magnitude (they are at least 1e-5
// after the clamp) and -1 <= bias <= 1 (a NaN difference makes the limited slope NaN
// by either division): then 2^-617 <= |r| <= 2^617, and the denominators 1 + r and
// (1 - bias) + (1 + bias) r of the positive-r branches lie in [2^-617, 2^619] with
// numerators 2 and 2r.

// d[k] *= limiter_value(num[k] / den[k]) for operands in that range and
// -1 <= bias <= 1, every piece computed and the right one selected.
template <int NF>
__device__ __forceinline__ void limited_slopes(const double (&num)[NF], const double (&den)[NF], double bias, int limiter,
                                               double (&d)[NF])
{
    double r[NF], R[NF];
#pragma unroll
    for (int k = 0; k < NF; k++) r[k] = div_in_range(num[k], den[k]);
#pragma unroll
    for (int k = 0; k < NF; k++) R[k] = r_coefficient(r[k], bias, InRangeDiv());   // used where r >= 0
    if (limiter == 0) {
#pragma unroll
        for (int k = 0; k < NF; k++) {
            const double hi = fmin(fmin(r[k], R[k]), 2.0);
            const double lo = (r[k] < 0.5) ? 2.0 * r[k] : 1.0;
            d[k] *= (r[k] < 0.0) ? 0.0 : ((r[k] < 1.0) ? lo : hi);
        }
    } else if (limiter == 1) {
#pragma unroll
        for (int k = 0; k < NF; k++) {
            const double v = fmin(div_in_range(2.0 * r[k], 1.0 + r[k]), R[k]);
            d[k] *= (r[k] < 0.0) ? 0.0 : v;
        }
    } else {
#pragma unroll
        for (int k = 0; k < NF; k++) {
            const double hi = fmin(1.0, R[k]);
            d[k] *= (r[k] < 0.0) ? 0.0 : ((r[k] < 1.0) ? r[k] : hi);
        }
    }
}

// limited_sides with IEEE divisions, for operands out of the short ones' range (no state
// the solvers reach) and for a bias outside [-1, 1], which they accept.  The fields are a loop over copies in scratch memory, so
// that this path adds little code to the kernels of many fields.
template <int NF, class NB>
__device__ __forceinline__ void limited_sides_any_range(const NB &UL, const double (&UM)[NF], const NB &UR, double bias,
                                                        int limiter, double (&xl)[NF], double (&xr)[NF])
{
    const double cl = 0.5 * (1.0 + bias), cr = 0.5 * (1.0 - bias);
    double l[NF], c[NF], r[NF];
#pragma unroll
    for (int k = 0; k < NF; k++) {
        l[k] = UL[k];
        c[k] = UM[k];
        r[k] = UR[k];
    }
#pragma clang loop unroll(disable)
    for (int k = 0; k < NF; k++) {
        const double dl = c[k] - l[k];
        const double dr = r[k] - c[k];
        double d = (cl * dl) + (cr * dr);
        const double num = (fabs(dl) < 1e-5) ? 1e-5 : dl;
        const double den = (fabs(dr) < 1e-5) ? 1e-5 : dr;
        d *= limiter_value(num / den, bias, limiter);
        l[k] = c[k] - (0.5 * d);
        r[k] = c[k] + (0.5 * d);
    }
#pragma unroll
    for (int k = 0; k < NF; k++) {
        xl[k] = l[k];
        xr[k] = r[k];
    }
}

// The middle cell's limited extrapolations to its two faces (EXACT).  Two cases need
// no division: slope differences of opposite signs (r < 0, the limiters' zero piece)
// and equal ones (r = 1 exactly, e.g. both clamped to 1e-5 in a flat region), whose
// limiter value is the same for every cell.  GROUP > 0: that many fields at a time,
// their division chains side by side (and no more slopes live at once); a wave all of
// whose cells and fields are such cases takes them, any other every piece of every
// field.  GROUP 0: branches, each lane taking its own pieces of a field at a time.
template <int NF, int GROUP, class NB>
__device__ __forceinline__ void limited_sides(const NB &UL, const double (&UM)[NF], const NB &UR, double bias, int limiter,
                                              double (&xl)[NF], double (&xr)[NF])
{
    const double cl = 0.5 * (1.0 + bias), cr = 0.5 * (1.0 - bias);
    double most = 0.0;
#pragma unroll
    for (int k = 0; k < NF; k++) most = fmax(fmax(most, fabs(UM[k] - UL[k])), fabs(UR[k] - UM[k]));
    if (!(most <= 0x1p600 && (bias >= -1.0) && (bias <= 1.0))) {
        limited_sides_any_range(UL, UM, UR, bias, limiter, xl, xr);
        return;
    }
    const double f1 = limiter_value(1.0, bias, limiter, InRangeDiv());
    if constexpr (GROUP == 0) {
#pragma unroll
        for (int k = 0; k < NF; k++) {
            const double dl = UM[k] - UL[k];
            const double dr = UR[k] - UM[k];
            double d = (cl * dl) + (cr * dr);
            const double num = (fabs(dl) < 1e-5) ? 1e-5 : dl;
            const double den = (fabs(dr) < 1e-5) ? 1e-5 : dr;
            double lim;
            if (num * den < 0.0) lim = 0.0;
            else if (num == den) lim = f1;
            else lim = limiter_value(div_in_range(num, den), bias, limiter, InRangeDiv());
            d *= lim;
            xl[k] = UM[k] - (0.5 * d);
            xr[k] = UM[k] + (0.5 * d);
        }
        return;
    }
    constexpr int N1 = GROUP > 0 ? GROUP : 1;
#pragma unroll
    for (int k0 = 0; k0 < NF; k0 += N1) {
        double num[N1], den[N1], d[N1];
        bool plain = true;
#pragma unroll
        for (int q = 0; q < N1; q++) {
            const int k = (k0 + q < NF) ? k0 + q : NF - 1;
            const double dl = UM[k] - UL[k];
            const double dr = UR[k] - UM[k];
            d[q] = (cl * dl) + (cr * dr);
            // |difference| < 1e-5 is replaced by +1e-5 (sign dropped) before the ratio.
            num[q] = (fabs(dl) < 1e-5) ? 1e-5 : dl;
            den[q] = (fabs(dr) < 1e-5) ? 1e-5 : dr;
            plain = plain && (num[q] * den[q] < 0.0 || num[q] == den[q]);
        }
        if (__all(plain)) {
#pragma unroll
            for (int q = 0; q < N1; q++) d[q] *= (num[q] == den[q]) ? f1 : 0.0;
        } else {
            limited_slopes(num, den, bias, limiter, d);
        }
#pragma unroll
        for (int q = 0; q < N1; q++) {
            if (k0 + q >= NF) continue;
            xl[k0 + q] = UM[k0 + q] - (0.5 * d[q]);
            xr[k0 + q] = UM[k0 + q] + (0.5 * d[q]);
        }
    }
}

// FAST-mode limiter: the same piecewise functions with Newton-refined reciprocals.
__device__ __forceinline__ double limiter_value_fast(double r, double bias, int limiter)
{
#pragma clang fp contract(on)
    if (r < 0.0) return 0.0;
    if (limiter == 0) {
        if (r < 0.5) return 2.0 * r;
        if (r < 1.0) return 1.0;
        return smin(smin(r, 2.0 * rcp_nr((1.0 - bias) + (1.0 + bias) * r)), 2.0);
    }
    if (limiter == 1) {
        const double R = 2.0 * rcp_nr((1.0 - bias) + (1.0 + bias) * r);
        return smin(2.0 * r * rcp_nr(1.0 + r), R);
    }
    if (r < 1.0) return r;
    return smin(1.0, 2.0 * rcp_nr((1.0 - bias) + (1.0 + bias) * r));
}

// Conserved state plus its physical flux in the sweep direction.
template <int NF>
struct ConsFlux {
    double U[NF];
    double F[NF];
};

// f(sl, sr, in_range) with the shared divisors of two densities: in_range is
// std::true_type, and the divisors are known to be fast, where both are in range and
// `also` holds.
template <class F>
__device__ __forceinline__ void with_divisors(double rho_l, double rho_r, bool also, const F &f)
{
    SharedDivisor sl = shared_divisor(rho_l), sr = shared_divisor(rho_r);
    if (sl.fast && sr.fast && also) {
        sl.fast = sr.fast = true;
        f(sl, sr, std::true_type{});
    } else {
        f(sl, sr, std::false_type{});
    }
}

// BRANCHES: the EXACT limiter by branches (each lane's pieces only) instead of by selects
// (every piece, the fields' chains side by side).  Branches for what fills the device:
// the walks of large grids up to nine fields, the batch kernel with many instances.
// EXACT, microseconds, branches / selects: 4 fields, x walk of 4096 x 4096 367 / 383, one
// 200 x 200 tile sweep 5.1 / 4.6; MHD 1024 x 1024 x tiles 67.7 / 61.9, y tiles 73.9 / 62.3,
// a step of 2300 x 2300 by walks 847 / 950 where one field varies, 1035 / 1071 where all
// do; HPR 1024 x 1024 y walk 183 / 164.
template <class P, int DIR, int MODE, bool BRANCHES = false>
struct Scheme {
    static constexpr int NF = P::NF;
    using Params = typename P::Params;

    __device__ static __forceinline__ void cons(const Params &m, const double (&w)[NF], double (&U)[NF])
    {
        if (MODE == MODE_EXACT) P::prim_to_cons(m, w, U);
        else P::prim_to_cons_fast(m, w, U);
    }

    // Flux of a conserved vector.
    __device__ static __forceinline__ void flux_of_cons(const Params &m, const double (&U)[NF], double (&F)[NF])
    {
        if (MODE == MODE_EXACT) {
            P::template flux<DIR>(m, U, F);
        } else {
            double w[NF];
            P::cons_to_prim_fast(m, U, w);
            P::template flux_prim_fast<DIR>(m, w, U, F);
        }
    }

    // Conserved vector and flux of a cell given as primitives.  EXACT: the
    // reference's state-overload flux, computeXFluxVector(computeConserved...)
    // (Euler/eulerstatevector.cpp:122-125).
    __device__ static __forceinline__ void cons_flux_of_prim(const Params &m, const double (&w)[NF], ConsFlux<NF> &cf)
    {
        cons(m, w, cf.U);
        if (MODE == MODE_EXACT) P::template flux<DIR>(m, cf.U, cf.F);
        else P::template flux_prim_fast<DIR>(m, w, cf.U, cf.F);
    }

    // MUSCL-Hancock half-step evolution of the middle cell's two boundary
    // extrapolations: SlopeLimiters::computeSlopeVector (slopelimiters.cpp:217-246)
    // then Solvers::evolveStateByHalfX/YTimeStep (Solvers/solvers.cpp:454-466,
    // 502-514) with computeEvolutionVector (:601-609) and evolveStateByHalfTimeStep
    // (:550-565).  Produces, for the SLIC face fluxes, the conserved vector and
    // flux of both evolved states: side 0 (left) and side 1 (right).
    // half_c = 0.5 * (ts / dx).
    __device__ static __forceinline__ void evolve(const Params &m, const double (&UL)[NF], const double (&UM)[NF],
                                                  const double (&UR)[NF], double bias, int limiter, double half_c,
                                                  ConsFlux<NF> &left, ConsFlux<NF> &right)
    {
        double xl[NF], xr[NF];
        const double cl = 0.5 * (1.0 + bias), cr = 0.5 * (1.0 - bias);
        if constexpr (MODE == MODE_EXACT) {
            limited_sides<NF, BRANCHES ? 0 : (NF <= 9 ? NF : 3)>(UL, UM, UR, bias, limiter, xl, xr);
            double Fl[NF], Fr[NF];
            if constexpr (HasSharedDivisor<P>::value) {
                // one branch for both sides, so their chains are scheduled together
                with_divisors(xl[0], xr[0], true, [&](const SharedDivisor &sl, const SharedDivisor &sr, auto) {
                    P::template flux_d<DIR>(m, xl, sl, Fl);
                    P::template flux_d<DIR>(m, xr, sr, Fr);
                });
            } else {
                flux_of_cons(m, xl, Fl);
                flux_of_cons(m, xr, Fr);
            }
#pragma unroll
            for (int k = 0; k < NF; k++) {
                const double evo = half_c * (Fl[k] - Fr[k]);
                xl[k] = xl[k] + evo;
                xr[k] = xr[k] + evo;
            }
        } else {
#pragma clang fp contract(on)
#pragma unroll
            for (int k = 0; k < NF; k++) {
                const double dl = UM[k] - UL[k];
                const double dr = UR[k] - UM[k];
                double d = (cl * dl) + (cr * dr);
                const double num = (fabs(dl) < 1e-5) ? 1e-5 : dl;
                const double den = (fabs(dr) < 1e-5) ? 1e-5 : dr;
                d *= limiter_value_fast(num * rcp_nr(den), bias, limiter);
                xl[k] = UM[k] - (0.5 * d);
                xr[k] = UM[k] + (0.5 * d);
            }
            double D[NF], Fr[NF];
            flux_of_cons(m, xr, Fr);
            if constexpr (HasFluxLess<P>::value) {
                double w[NF];
                P::cons_to_prim_fast(m, xl, w);
                P::template flux_less_fast<DIR>(m, w, xl, Fr, D);
            } else {
                flux_of_cons(m, xl, D);
#pragma unroll
                for (int k = 0; k < NF; k++) D[k] = D[k] - Fr[k];
            }
#pragma unroll
            for (int k = 0; k < NF; k++) {
                xl[k] = xl[k] + half_c * D[k];
                xr[k] = xr[k] + half_c * D[k];
            }
        }
        if (MODE == MODE_EXACT) {
            // setConservedVariableVector, then the FORCE flux converts the state
            // back: computeConservedVariableVector + state-overload flux.  The
            // round trip returns rho unchanged, so the way back and the flux divide
            // by the density whose reciprocal the way out already holds.
            double w[NF];
            if constexpr (HasSharedDivisor<P>::value) {
                with_divisors(xl[0], xr[0], scale_in_range(m.gm1),
                              [&](const SharedDivisor &sl, const SharedDivisor &sr, auto in_range) {
                                  double wr[NF];
                                  P::cons_to_prim_d(m, xl, sl, w);
                                  P::cons_to_prim_d(m, xr, sr, wr);
                                  if constexpr (decltype(in_range)::value) {
                                      P::prim_to_cons_d(m, w, sl, left.U);
                                      P::prim_to_cons_d(m, wr, sr, right.U);
                                  } else {
                                      cons(m, w, left.U);
                                      cons(m, wr, right.U);
                                  }
                                  P::template flux_d<DIR>(m, left.U, sl, left.F);
                                  P::template flux_d<DIR>(m, right.U, sr, right.F);
                              });
            } else if constexpr (HasRoundTrip<P>::value) {
                P::template round_trip<DIR>(m, xl, left.U, left.F);
                P::template round_trip<DIR>(m, xr, right.U, right.F);
            } else {
                P::cons_to_prim(m, xl, w);
                cons_flux_of_prim(m, w, left);
                P::cons_to_prim(m, xr, w);
                cons_flux_of_prim(m, w, right);
            }
        } else {
            double w[NF];
#pragma unroll
            for (int k = 0; k < NF; k++) { left.U[k] = xl[k]; right.U[k] = xr[k]; }
            P::cons_to_prim_fast(m, xl, w);
            P::template flux_prim_fast<DIR>(m, w, left.U, left.F);
            P::cons_to_prim_fast(m, xr, w);
            P::template flux_prim_fast<DIR>(m, w, right.U, right.F);
        }
    }

    // FORCE flux between two states: FirstOrderSolver::computeLaxFriedrichsFlux
    // (firstordersolver.cpp:79-85), computeRichtmyerFlux (:165-171) followed by the
    // flux of the intermediate state (:96-97), and computeFORCEFlux (:227-230).
    // lf_c = dx / ts, ri_c = ts / dx.
    __device__ static __forceinline__ void force_face(const Params &m, const ConsFlux<NF> &a, const ConsFlux<NF> &b,
                                                      double lf_c, double ri_c, double (&F)[NF])
    {
        double us[NF], lf[NF], ri[NF];
        if constexpr (MODE == MODE_EXACT) {
#pragma unroll
            for (int k = 0; k < NF; k++) {
                lf[k] = 0.5 * ((a.F[k] + b.F[k]) + (lf_c * (a.U[k] - b.U[k])));
                us[k] = 0.5 * ((a.U[k] + b.U[k]) + (ri_c * (a.F[k] - b.F[k])));
            }
            flux_of_cons(m, us, ri);
#pragma unroll
            for (int k = 0; k < NF; k++) F[k] = 0.5 * (lf[k] + ri[k]);
        } else {
#pragma clang fp contract(on)
#pragma unroll
            for (int k = 0; k < NF; k++) {
                lf[k] = (a.F[k] + b.F[k]) + lf_c * (a.U[k] - b.U[k]);
                us[k] = 0.5 * ((a.U[k] + b.U[k]) + ri_c * (a.F[k] - b.F[k]));
            }
            flux_of_cons(m, us, ri);
#pragma unroll
            for (int k = 0; k < NF; k++) F[k] = 0.5 * (0.5 * lf[k] + ri[k]);   // the half fused into the sum
        }
    }

    // FirstOrderSolver::computeFORCEUpdate (firstordersolver.cpp:428-433) followed
    // by setConservedVariableVector.  up_c = ts / dx.
    __device__ static __forceinline__ void update(const Params &m, const double (&U)[NF], const double (&Fm)[NF],
                                                  const double (&Fp)[NF], double up_c, double (&w)[NF])
    {
        double N[NF];
        if constexpr (MODE == MODE_EXACT) {
#pragma unroll
            for (int k = 0; k < NF; k++) N[k] = U[k] + (up_c * (Fm[k] - Fp[k]));
            P::cons_to_prim(m, N, w);
        } else {
#pragma clang fp contract(on)
#pragma unroll
            for (int k = 0; k < NF; k++) N[k] = U[k] + (up_c * (Fm[k] - Fp[k]));
            P::cons_to_prim_fast(m, N, w);
        }
    }
};

}  // namespace vg
