// mfc_device.hpp -- per-cell and per-face device arithmetic of the RHS.
//
// Every routine restates the reference's arithmetic in its evaluation order
// (the plain units are built with -ffp-contract=off, so each multiply and add
// is rounded on its own, like the Fortran statements).  R is the arithmetic
// type of the WENO/HLLC bulk: double for the FP64 forms, float for the
// FP32-bulk form.  Conversion to primitive variables always runs in double.
//
// The arithmetic lives in an inline namespace named by the translation unit's
// form (MFC_FORM), so units built with different flags or with the
// contracted FP64 form (MFC_FAST_F64 = 1: FMA contraction, divisions as a
// multiply by a Newton-refined reciprocal, the WENO weights normalised by one
// reciprocal of their sum, square roots from v_rsq_f64 refined) never share
// a kernel or function symbol.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#ifndef MFC_FORM
#define MFC_FORM ieee
#endif
#ifndef MFC_FAST_F64
#define MFC_FAST_F64 0
#endif

namespace mfc {

constexpr int kNumFluidsMax = 10;
constexpr int kMaxSys = 2 * kNumFluidsMax + 3 + 1;

// Index layout of the 5-equation system (m_global_parameters.fpp:302-310):
// [alpha_i rho_i (NF), momentum (D), E, alpha_i (NF)], 0-based.
template <int NF, int D>
struct Sys {
    static constexpr int S = 2 * NF + D + 1;
    static constexpr int MOM = NF;
    static constexpr int E = NF + D;
    static constexpr int ADV = NF + D + 1;
};

struct Eos {
    double gammas[kNumFluidsMax];
    double pi_infs[kNumFluidsMax];
};

// WENO coefficient planes of the 27-entry table: poly_coef_cbL(r,q) at
// 2r+q, cbR at 6+2r+q, d_cbL(r) at 12+r, d_cbR(r) at 15+r, beta_coef(r,q) at
// 18+3r+q.
enum { kCbL = 0, kCbR = 6, kDL = 12, kDR = 15, kBeta = 18, kNCoef = 27 };

// Kinds of WENO5 coefficients a kernel is built for: each cell's own from the
// table; one set for every cell, in scalar registers; and in the contracted
// form those of cells of equal width, built in (weno5_canon).
enum CoefKind { kCellCoef = 0, kEqualCoef = 1, kCanonCoef = 2 };

inline namespace MFC_FORM {

constexpr bool kFastF64 = MFC_FAST_F64 != 0;

// Reciprocal of an FP64 value to within about one ulp: v_rcp_f64 (relative
// error e of about 2^-24) refined by one third-order step, r (1 + e + e^2),
// whose own error is e^3: three FMAs where two Newton steps take four.
// Valid where b and 1/b are normal; 0 and infinities give NaN.
__device__ __forceinline__ double frcp(double b) {
    const double r = __builtin_amdgcn_rcp(b);
    const double e = __builtin_fma(-b, r, 1.0);
    return __builtin_fma(r, __builtin_fma(e, e, e), r);
}

// Square root to within about one ulp from v_rsq_f64 (5e-8 relative): one
// Newton step on the reciprocal square root, then one on the root itself.
// 0 gives 0 and a negative argument NaN, like sqrt; no range scaling, so
// arguments below 1e-290 are not handled (the squared sound speeds it takes
// are far above that).
__device__ __forceinline__ double fsqrt(double x) {
    const double y0 = __builtin_amdgcn_rsq(x);
    const double y1 = __builtin_fma(y0, __builtin_fma(-0.5 * x * y0, y0, 0.5), y0);
    const double g = x * y1;
    const double r = __builtin_fma(-g, g, x);
    const double root = __builtin_fma(0.5 * y1, r, g);
    return x == 0.0 ? x : root;
}

// Division in the bulk precision: IEEE correctly rounded in the plain FP64
// form (it reproduces the reference bit for bit); a multiply by frcp (about
// 1.5 ulp) in the contracted FP64 form; in the FP32 bulk a reciprocal-multiply
// (about 1 ulp), which is what that form trades for speed.
__device__ __forceinline__ double bdiv(double a, double b) {
    if constexpr (kFastF64)
        return a * frcp(b);
    else
        return a / b;
}
__device__ __forceinline__ float bdiv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ double bsqrt(double a) {
    if constexpr (kFastF64)
        return fsqrt(a);
    else
        return sqrt(a);
}
__device__ __forceinline__ float bsqrt(float a) { return __builtin_amdgcn_sqrtf(a); }

template <typename T>
__device__ __forceinline__ T min_ref(T a, T b) { return (a < b) ? a : b; }
template <typename T>
__device__ __forceinline__ T max_ref(T a, T b) { return (a > b) ? a : b; }

// Conservative -> primitive at one cell:
// m_variables_conversion.fpp:329-370 with the mixture rule of :199-207 and
// the pressure of :98-106.  rho is clamped at sgm_eps = 1e-16 (:353).
template <int NF, int D>
__device__ __forceinline__ void cons_to_prim(const double *c, double *p, const Eos &eos) {
    using Y = Sys<NF, D>;
    double rho = 0.0, gam = 0.0, pinf = 0.0, dyn = 0.0;
#pragma unroll
    for (int i = 0; i < NF; ++i) p[i] = c[i];
#pragma unroll
    for (int i = 0; i < NF; ++i) {
        rho = rho + c[i];
        gam = gam + c[Y::ADV + i] * eos.gammas[i];
        pinf = pinf + c[Y::ADV + i] * eos.pi_infs[i];
    }
    rho = max_ref(rho, 1e-16);
    if constexpr (kFastF64) {
        // 1/rho and 1/Gamma from one reciprocal of their product
        const double r = frcp(rho * gam), irho = gam * r, igam = rho * r;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            p[Y::MOM + d] = c[Y::MOM + d] * irho;
            dyn = dyn + 0.5 * c[Y::MOM + d] * p[Y::MOM + d];
        }
        p[Y::E] = (c[Y::E] - dyn - pinf) * igam;
    } else {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            p[Y::MOM + d] = bdiv(c[Y::MOM + d], rho);
            dyn = dyn + 0.5 * c[Y::MOM + d] * p[Y::MOM + d];
        }
        p[Y::E] = bdiv(c[Y::E] - dyn - pinf, gam);
    }
#pragma unroll
    for (int i = 0; i < NF; ++i) p[Y::ADV + i] = c[Y::ADV + i];
}

// FP64 quotient of the WENO weights: the instruction sequence the compiler
// emits for an IEEE a / b on gfx950 (v_rcp_f64, two Newton steps, the
// quotient and one residual correction) without its range-scaling
// (v_div_scale) and special-case (v_div_fixup) steps.  Those steps change
// nothing -- the result is the correctly rounded quotient, bit for bit
// a / b -- when b, 1/b and a/b are normal, |a| >= 2^-969 (or a = 0) and the
// exponents of a and b differ by less than 768.  For the weights this holds
// whenever every squared smoothness indicator beta^2 lies in [1e-200, 1e100]:
// alpha = d/beta^2 with ideal weights d in [1e-3, 1] is then in [1e-103,
// 1e200] and omega = alpha/sum(alpha) >= 3e-304.  beta >= weno_eps >= 1e-100
// (checked by mfc_rhs_init) gives the lower end; the upper end, beta <= 1e50,
// holds for any stencil whose differences are below ~1e24, i.e. for every
// physical state (a diverging run reaches inf/NaN, which both divisions
// propagate, and the NaN guard stops it).
__device__ __forceinline__ double ndiv(double a, double b) {
    const double r = __builtin_amdgcn_rcp(b);
    const double e0 = __builtin_fma(-b, r, 1.0);
    const double r1 = __builtin_fma(r, e0, r);
    const double e1 = __builtin_fma(-b, r1, 1.0);
    const double r2 = __builtin_fma(r1, e1, r1);
    const double q = a * r2;
    const double rem = __builtin_fma(-b, q, a);
    return __builtin_fma(rem, r2, q);
}

template <bool FAST>
__device__ __forceinline__ double wdiv(double a, double b) {
    if constexpr (FAST)
        return ndiv(a, b);
    else
        return a / b;
}
template <bool FAST>
__device__ __forceinline__ float wdiv(float a, float b) {
    return bdiv(a, b);
}

// Reconstruction of one variable at one cell (m_weno.fpp:391-540): v[0..WO-1]
// is the stencil j-polyn..j+polyn, cf the cell's coefficients.  Computes the
// smoothness indicators once and evaluates the left (face j-1/2) and/or right
// (face j+1/2) value (smoothness indicators m_weno.fpp:476-506, WENO3
// :425-438).  In the plain FP64 form the weight divisions are ndiv
// (bit-identical to IEEE division in the range stated there); the contracted
// form multiplies by the reciprocals of beta_k^2 and of sum(alpha), which
// both faces share.
template <int WO, typename R, bool WANT_L, bool WANT_R>
__device__ __forceinline__ void weno_cell(const R *v, const R *cf, R eps, R &vL, R &vR) {
    if constexpr (WO == 1) {
        vL = v[0];
        vR = v[0];
    } else if constexpr (WO == 3) {
        const R vj = v[1];
        const R d0 = v[2] - v[1], dm1 = v[1] - v[0];
        const R b0 = cf[kBeta + 0] * d0 * d0 + eps;
        const R b1 = cf[kBeta + 3] * dm1 * dm1 + eps;
        const R bb0 = b0 * b0, bb1 = b1 * b1;
        const R pL0 = vj + cf[kCbL + 0] * d0, pL1 = vj + cf[kCbL + 2] * dm1;
        const R pR0 = vj + cf[kCbR + 0] * d0, pR1 = vj + cf[kCbR + 2] * dm1;
        if constexpr (kFastF64 && sizeof(R) == 8) {
            // omega_k = alpha_k / sum(alpha) with alpha_k = d_k / beta_k^2 is
            // unchanged when every alpha is multiplied by beta_0^2 beta_1^2:
            // alpha'_k = d_k * (the other beta^2), and one reciprocal of the
            // sum per face
            if constexpr (WANT_L) {
                const R a0 = cf[kDL + 0] * bb1, a1 = cf[kDL + 1] * bb0;
                vL = (a0 * pL0 + a1 * pL1) * frcp(a0 + a1);
            }
            if constexpr (WANT_R) {
                const R a0 = cf[kDR + 0] * bb1, a1 = cf[kDR + 1] * bb0;
                vR = (a0 * pR0 + a1 * pR1) * frcp(a0 + a1);
            }
            return;
        }
        auto weights = [&](auto fast) {
            constexpr bool F = decltype(fast)::value;
            if constexpr (WANT_L) {
                const R a0 = wdiv<F>(cf[kDL + 0], bb0);
                const R a1 = wdiv<F>(cf[kDL + 1], bb1);
                const R s = a0 + a1;
                vL = wdiv<F>(a0, s) * pL0 + wdiv<F>(a1, s) * pL1;
            }
            if constexpr (WANT_R) {
                const R a0 = wdiv<F>(cf[kDR + 0], bb0);
                const R a1 = wdiv<F>(cf[kDR + 1], bb1);
                const R s = a0 + a1;
                vR = wdiv<F>(a0, s) * pR0 + wdiv<F>(a1, s) * pR1;
            }
        };
        weights(std::integral_constant<bool, sizeof(R) == 8>{});
    } else {
        const R vj = v[2];
        const R d1 = v[4] - v[3], d0 = v[3] - v[2], dm1 = v[2] - v[1], dm2 = v[1] - v[0];
        R b0, b1, b2;
        if constexpr ((kFastF64 && sizeof(R) == 8) || sizeof(R) == 4) {
            // contracted forms: c0 a^2 + c1 a b + c2 b^2 + eps as
            // a (c0 a + c1 b) + (c2 b b + eps), five operations where the
            // reference's order takes seven
            auto beta = [&](R c0, R c1, R c2, R a, R b) {
                return __builtin_fma(a, __builtin_fma(c1, b, c0 * a), __builtin_fma(c2 * b, b, eps));
            };
            b0 = beta(cf[kBeta + 0], cf[kBeta + 1], cf[kBeta + 2], d1, d0);
            b1 = beta(cf[kBeta + 3], cf[kBeta + 4], cf[kBeta + 5], d0, dm1);
            b2 = beta(cf[kBeta + 6], cf[kBeta + 7], cf[kBeta + 8], dm1, dm2);
        } else {
            b0 = cf[kBeta + 0] * d1 * d1 + cf[kBeta + 1] * d1 * d0 + cf[kBeta + 2] * d0 * d0 + eps;
            b1 = cf[kBeta + 3] * d0 * d0 + cf[kBeta + 4] * d0 * dm1 + cf[kBeta + 5] * dm1 * dm1 + eps;
            b2 = cf[kBeta + 6] * dm1 * dm1 + cf[kBeta + 7] * dm1 * dm2 + cf[kBeta + 8] * dm2 * dm2 + eps;
        }
        const R bb0 = b0 * b0, bb1 = b1 * b1, bb2 = b2 * b2;
        R pL[3], pR[3];
        if constexpr (WANT_L) {
            pL[0] = vj + cf[kCbL + 0] * d1 + cf[kCbL + 1] * d0;
            pL[1] = vj + cf[kCbL + 2] * d0 + cf[kCbL + 3] * dm1;
            pL[2] = vj + cf[kCbL + 4] * dm1 + cf[kCbL + 5] * dm2;
        }
        if constexpr (WANT_R) {
            pR[0] = vj + cf[kCbR + 0] * d1 + cf[kCbR + 1] * d0;
            pR[1] = vj + cf[kCbR + 2] * d0 + cf[kCbR + 3] * dm1;
            pR[2] = vj + cf[kCbR + 4] * dm1 + cf[kCbR + 5] * dm2;
        }
        if constexpr (kFastF64 && sizeof(R) == 8) {
            // the weights scaled by beta_0^2 beta_1^2 beta_2^2 (the ratios are
            // unchanged): alpha'_k = d_k * the product of the other two
            // beta^2, no reciprocal per candidate (weno_eps >= 1e-50 keeps
            // the products normal)
            const R q12 = bb1 * bb2, q02 = bb0 * bb2, q01 = bb0 * bb1;
            if constexpr (WANT_L && WANT_R) {
                // both faces' normalisations from one reciprocal of the
                // product of the two sums
                const R a0 = cf[kDL + 0] * q12, a1 = cf[kDL + 1] * q02, a2 = cf[kDL + 2] * q01;
                const R b0 = cf[kDR + 0] * q12, b1 = cf[kDR + 1] * q02, b2 = cf[kDR + 2] * q01;
                const R sL = a0 + a1 + a2, sR = b0 + b1 + b2;
                const R r = frcp(sL * sR);
                vL = (a0 * pL[0] + a1 * pL[1] + a2 * pL[2]) * (sR * r);
                vR = (b0 * pR[0] + b1 * pR[1] + b2 * pR[2]) * (sL * r);
            } else if constexpr (WANT_L) {
                const R a0 = cf[kDL + 0] * q12, a1 = cf[kDL + 1] * q02, a2 = cf[kDL + 2] * q01;
                vL = (a0 * pL[0] + a1 * pL[1] + a2 * pL[2]) * frcp(a0 + a1 + a2);
            } else if constexpr (WANT_R) {
                const R a0 = cf[kDR + 0] * q12, a1 = cf[kDR + 1] * q02, a2 = cf[kDR + 2] * q01;
                vR = (a0 * pR[0] + a1 * pR[1] + a2 * pR[2]) * frcp(a0 + a1 + a2);
            }
            return;
        }
        auto weights = [&](auto fast) {
            constexpr bool F = decltype(fast)::value;
            if constexpr (WANT_L) {
                const R a0 = wdiv<F>(cf[kDL + 0], bb0), a1 = wdiv<F>(cf[kDL + 1], bb1),
                        a2 = wdiv<F>(cf[kDL + 2], bb2);
                const R s = a0 + a1 + a2;
                vL = wdiv<F>(a0, s) * pL[0] + wdiv<F>(a1, s) * pL[1] + wdiv<F>(a2, s) * pL[2];
            }
            if constexpr (WANT_R) {
                const R a0 = wdiv<F>(cf[kDR + 0], bb0), a1 = wdiv<F>(cf[kDR + 1], bb1),
                        a2 = wdiv<F>(cf[kDR + 2], bb2);
                const R s = a0 + a1 + a2;
                vR = wdiv<F>(a0, s) * pR[0] + wdiv<F>(a1, s) * pR[1] + wdiv<F>(a2, s) * pR[2];
            }
        };
        weights(std::integral_constant<bool, sizeof(R) == 8>{});
    }
}

// Both faces of a WENO5 cell on a grid of equal widths, contracted form: the
// coefficients are the constants of the uniform grid, so the arithmetic can
// be arranged for them.  Smoothness indicators times 3/4 (the weights do not
// change when eps is scaled too) have unit leading coefficients and share
// the squares of the two inner differences; the ideal weights times 10 are
// (3, 6, 1) and (1, 6, 3), so one candidate of each side takes its product
// of squares as it is; the candidates enter as three times their deviation
// from the cell value, one FMA each, and the cell value is added last, so
// the rounding of the normalisation scales with the deviation instead of
// with the value.  50 FP64 operations and a reciprocal instead of 62 in the
// general form above; the sweeps are bound by VALU issue: 512^3 droplet x and
// y sweep 9.13 -> 8.35 ms, z 5.59 -> 5.45 ms per launch, step 44.8 -> 42.1 ms,
// 768^2 x and y sweep 47 -> 40 us.
// The constants that are no inline operands are kept in scalar registers:
// as literals they go through fmac instructions, whose addend must first be
// copied (about 6 moves per call).
struct CanonK {
    double c275 = 2.75, c25 = 2.5, c125 = 1.25, c15 = 1.5, c6 = 6.0, c18 = 18.0;
    __device__ __forceinline__ CanonK() { asm("" : "+s"(c275), "+s"(c25), "+s"(c125), "+s"(c15), "+s"(c6), "+s"(c18)); }
};
__device__ __forceinline__ void weno5_canon(const double *v, double eps, double &vL, double &vR, const CanonK &K) {
    const double d1 = v[4] - v[3], d0 = v[3] - v[2], dm1 = v[2] - v[1], dm2 = v[1] - v[0];
    const double e = 0.75 * eps, P0 = d0 * d0, Pm = dm1 * dm1;
    const double b0 = __builtin_fma(d1, __builtin_fma(-K.c275, d0, d1), __builtin_fma(K.c25, P0, e));
    const double b1 = __builtin_fma(d0, __builtin_fma(-K.c125, dm1, d0), Pm + e);
    const double b2 = __builtin_fma(dm2, __builtin_fma(-K.c275, dm1, dm2), __builtin_fma(K.c25, Pm, e));
    const double bb0 = b0 * b0, bb1 = b1 * b1, bb2 = b2 * b2;
    const double q12 = bb1 * bb2, q02 = bb0 * bb2, q01 = bb0 * bb1;
    const double m = K.c6 * q02, M = K.c18 * q02, y0 = K.c15 * q12, y2 = K.c15 * q01;
    const double sR = __builtin_fma(K.c6, y0, __builtin_fma(2.0, y2, M));
    const double sL = __builtin_fma(2.0, y0, __builtin_fma(K.c6, y2, M));
    const double nR = __builtin_fma(y0, __builtin_fma(4.0, d0, -d1),
                                    __builtin_fma(m, __builtin_fma(0.5, dm1, d0), q01 * __builtin_fma(K.c25, dm1, -dm2)));
    const double nL = __builtin_fma(y2, __builtin_fma(-4.0, dm1, dm2),
                                    __builtin_fma(-m, __builtin_fma(0.5, d0, dm1), q12 * __builtin_fma(-K.c25, d0, d1)));
    const double r = frcp(sL * sR);
    vL = __builtin_fma(nL, sR * r, v[2]);
    vR = __builtin_fma(nR, sL * r, v[2]);
}

// Both faces of one cell, as the kernels of a coefficient kind (UNI, a
// CoefKind) reconstruct them.
template <int WO, typename R, int UNI>
__device__ __forceinline__ void weno_both(const R *v, const R *cf, R eps, R &vL, R &vR, const CanonK &K) {
    if constexpr (UNI == kCanonCoef) {
        static_assert(kFastF64 && sizeof(R) == 8 && WO == 5, "contracted form");
        weno5_canon(v, eps, vL, vR, K);
    } else {
        weno_cell<WO, R, true, true>(v, cf, eps, vL, vR);
    }
}

// HLLC flux at one face, normal direction DIR
// (m_riemann_solvers.fpp:134-325).  qL is the state left of the face (the
// right-face reconstruction of the left cell), qR the state right of it.
// flux[] gets sys_size values, ustar the contact velocity that drives the
// alpha*div(u) source.  With VSRC, vsrc[0..D-1] receives every component of
// that star-region velocity, vel_src_rs (:313-323), which the viscous energy
// flux multiplies.
template <int NF, int D, int DIR, typename R, bool VSRC = false>
__device__ __forceinline__ void hllc_face(const R *qL, const R *qR, const Eos &eos, R *flux, R &ustar,
                                          R *vsrc = nullptr) {
    using Y = Sys<NF, D>;
    R vel_L_rms = R(0), vel_R_rms = R(0);
#pragma unroll
    for (int d = 0; d < D; ++d) {
        vel_L_rms = vel_L_rms + qL[Y::MOM + d] * qL[Y::MOM + d];
        vel_R_rms = vel_R_rms + qR[Y::MOM + d] * qR[Y::MOM + d];
    }
    const R pres_L = qL[Y::E], pres_R = qR[Y::E];
    R rho_L = R(0), gamma_L = R(0), pi_inf_L = R(0);
    R rho_R = R(0), gamma_R = R(0), pi_inf_R = R(0);
#pragma unroll
    for (int i = 0; i < NF; ++i) {
        rho_L = rho_L + qL[i];
        gamma_L = gamma_L + qL[Y::ADV + i] * R(eos.gammas[i]);
        pi_inf_L = pi_inf_L + qL[Y::ADV + i] * R(eos.pi_infs[i]);
        rho_R = rho_R + qR[i];
        gamma_R = gamma_R + qR[Y::ADV + i] * R(eos.gammas[i]);
        pi_inf_R = pi_inf_R + qR[Y::ADV + i] * R(eos.pi_infs[i]);
    }
    const R E_L = gamma_L * pres_L + pi_inf_L + R(0.5) * rho_L * vel_L_rms;
    const R E_R = gamma_R * pres_R + pi_inf_R + R(0.5) * rho_R * vel_R_rms;
    R c_L, c_R;
    if constexpr (kFastF64 && sizeof(R) == 8) {
        // c^2 = (H - |u|^2/2)/Gamma = (E + p - rho |u|^2/2)/(rho Gamma), both
        // sides from one reciprocal of the product of their denominators
        const R gL = rho_L * gamma_L, gR = rho_R * gamma_R;
        const R rg = frcp(gL * gR);
        c_L = bsqrt((E_L + pres_L - R(0.5) * rho_L * vel_L_rms) * (gR * rg));
        c_R = bsqrt((E_R + pres_R - R(0.5) * rho_R * vel_R_rms) * (gL * rg));
    } else {
        const R H_L = bdiv(E_L + pres_L, rho_L);
        const R H_R = bdiv(E_R + pres_R, rho_R);
        c_L = bsqrt(bdiv(H_L - R(0.5) * vel_L_rms, gamma_L));
        c_R = bsqrt(bdiv(H_R - R(0.5) * vel_R_rms, gamma_R));
    }
    const R uL = qL[Y::MOM + DIR], uR = qR[Y::MOM + DIR];
    const R s_L = min_ref(uL - c_L, uR - c_R);
    const R s_R = max_ref(uR + c_R, uL + c_L);
    const R s_S = bdiv(pres_R - pres_L + rho_L * uL * (s_L - uL) - rho_R * uR * (s_R - uR),
                       rho_L * (s_L - uL) - rho_R * (s_R - uR));
    const R s_M = min_ref(R(0), s_L);
    const R s_P = max_ref(R(0), s_R);
    if constexpr (((kFastF64 && sizeof(R) == 8) || sizeof(R) == 4) && !VSRC) {
        // The weights xi_M = 1/2 + sign(1/2, s_S) and xi_P = 1/2 - sign(1/2,
        // s_S) below are 1 and 0 or 0 and 1 by the sign bit of s_S, so for
        // finite states the flux is the upwind side's expression and the
        // other side adds exact zeros.  The contracted forms evaluate the
        // upwind side only; the contact velocity is then its m.
        const bool lft = !signbit(s_S);
        const R rho = lft ? rho_L : rho_R, u = lft ? uL : uR, p = lft ? pres_L : pres_R, E = lft ? E_L : E_R;
        const R sw = lft ? s_L : s_R, sm = lft ? s_M : s_P;
        R xi, pd; // (s - u)/(s - s_S), p/(s - u)
        if constexpr (kFastF64 && sizeof(R) == 8) {
            // both from one reciprocal of (s - u)(s - s_S)
            const R du = sw - u, ds = sw - s_S;
            const R r = frcp(du * ds);
            xi = du * du * r;
            pd = p * ds * r;
        } else {
            xi = bdiv(sw - u, sw - s_S);
            pd = bdiv(p, sw - u);
        }
        const R m = u + sm * (xi - R(1));
#pragma unroll
        for (int i = 0; i < NF; ++i) flux[i] = (lft ? qL[i] : qR[i]) * m;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const R v = lft ? qL[Y::MOM + d] : qR[Y::MOM + d];
            if (d == DIR)
                flux[Y::MOM + d] = rho * (u * v + sm * (xi * s_S - v)) + p;
            else
                flux[Y::MOM + d] = rho * (u * v + sm * (xi * v - v));
        }
        flux[Y::E] = u * (E + p) + sm * (xi * (E + (s_S - u) * (rho * s_S + pd)) - E);
#pragma unroll
        for (int i = 0; i < NF; ++i) flux[Y::ADV + i] = (lft ? qL[Y::ADV + i] : qR[Y::ADV + i]) * m;
        ustar = m;
        return;
    }
    // 1/(s_L - u_L), 1/(s_R - u_R), 1/(s_L - s_S), 1/(s_R - s_S): in the
    // contracted form from one reciprocal of their product
    R xi_L, xi_R, iwL = R(0), iwR = R(0);
    if constexpr (kFastF64 && sizeof(R) == 8) {
        const R dL = s_L - uL, dR = s_R - uR, eL = s_L - s_S, eR = s_R - s_S;
        const R pd = dL * dR, pe = eL * eR;
        const R r4 = frcp(pd * pe);
        xi_L = dL * (pd * eR * r4);
        xi_R = dR * (pd * eL * r4);
        iwL = dR * pe * r4;
        iwR = dL * pe * r4;
    } else {
        xi_L = bdiv(s_L - uL, s_L - s_S);
        xi_R = bdiv(s_R - uR, s_R - s_S);
    }
    // Fortran sign(0.5, s_S) takes the sign bit of s_S, so -0.0 gives -0.5.
    const R hs = copysign(R(0.5), s_S);
    const R xi_M = (R(0.5) + hs);
    const R xi_P = (R(0.5) - hs);
    const R mL = uL + s_M * (xi_L - R(1));
    const R mR = uR + s_P * (xi_R - R(1));
#pragma unroll
    for (int i = 0; i < NF; ++i) flux[i] = xi_M * qL[i] * mL + xi_P * qR[i] * mR;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const R flg = (d == DIR) ? R(1) : R(0);
        const R vLd = qL[Y::MOM + d], vRd = qR[Y::MOM + d];
        flux[Y::MOM + d] =
            xi_M * (rho_L * (uL * vLd + s_M * (xi_L * (flg * s_S + (R(1) - flg) * vLd) - vLd)) + flg * (pres_L)) +
            xi_P * (rho_R * (uR * vRd + s_P * (xi_R * (flg * s_S + (R(1) - flg) * vRd) - vRd)) + flg * (pres_R));
    }
    R pdL, pdR; // p_L/(s_L - u_L), p_R/(s_R - u_R)
    if constexpr (kFastF64 && sizeof(R) == 8) {
        pdL = pres_L * iwL;
        pdR = pres_R * iwR;
    } else {
        pdL = bdiv(pres_L, s_L - uL);
        pdR = bdiv(pres_R, s_R - uR);
    }
    flux[Y::E] = xi_M * (uL * (E_L + pres_L) + s_M * (xi_L * (E_L + (s_S - uL) * (rho_L * s_S + pdL)) - E_L)) +
                 xi_P * (uR * (E_R + pres_R) + s_P * (xi_R * (E_R + (s_S - uR) * (rho_R * s_S + pdR)) - E_R));
#pragma unroll
    for (int i = 0; i < NF; ++i) flux[Y::ADV + i] = xi_M * qL[Y::ADV + i] * mL + xi_P * qR[Y::ADV + i] * mR;
    // dir_flg = 1 for the normal component: xi_M*(u_L + 1*s_M*(xi_L-1)) + ...
    ustar = xi_M * (uL + R(1) * s_M * (xi_L - R(1))) + xi_P * (uR + R(1) * s_P * (xi_R - R(1)));
    if constexpr (VSRC) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const R flg = (d == DIR) ? R(1) : R(0);
            vsrc[d] = xi_M * (qL[Y::MOM + d] + flg * s_M * (xi_L - R(1))) +
                      xi_P * (qR[Y::MOM + d] + flg * s_P * (xi_R - R(1)));
        }
    }
}

} // inline namespace MFC_FORM
} // namespace mfc
