// hf_physics.h -- per-cell and per-face arithmetic of the Euler step for gfx950.
//
// Every expression keeps the reference's evaluation order (binary64 with the
// FP64 policy, compiled with -ffp-contract=off), so the FP64 kernels are
// bit-identical to the reference CPU path.  Paths below are relative to the
// reference checkout under src/fvm_2d_cart/.
//
// Deliberate, bit-preserving differences from the reference's code shape:
//  * primitives, E and the sound speed of a state are computed once and
//    shared by its flux and the HLLC star state (same formula, same operands);
//  * HLLC evaluates only the star state of the selected branch;
//  * the limiters evaluate one division (a correctly rounded quotient is
//    monotone in the numerator, so min(2r/(1+r), 2/(1+r)) = min(2r,2)/(1+r)).
#pragma once
#include <hip/hip_runtime.h>

namespace hf {

// Exact binary64: IEEE division and the correctly rounded square root.
struct MathF64 {
    typedef double R;
    static __device__ __forceinline__ double div(double a, double b) { return a / b; }
    static __device__ __forceinline__ double sqrt(double x) { return __builtin_sqrt(x); }
    static __device__ __forceinline__ double fabs(double x) { return __builtin_fabs(x); }
    static constexpr double tol = 1e-6;
    static constexpr bool fast = false;   // the reference's expressions, in its order
};

// Bulk FP32: hardware reciprocal and square root (about 1 ulp each).
struct MathF32 {
    typedef float R;
    static __device__ __forceinline__ float div(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
    static __device__ __forceinline__ float sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
    static __device__ __forceinline__ float fabs(float x) { return __builtin_fabsf(x); }
    static constexpr float tol = 1e-6f;
    static constexpr bool fast = true;    // the FP32 formulation of namespace f32 below
};

// std::min / std::max (NaN handling of the reference:
// scheme/riemann/riemann_hllc/riemann_hllc.cpp:146-147, timestep.cpp:51-52).
template <class R> __device__ __forceinline__ R smin(R a, R b) { return (b < a) ? b : a; }
template <class R> __device__ __forceinline__ R smax(R a, R b) { return (a < b) ? b : a; }

// A conserved state with its primitives, total energy (re-derived from the
// primitives) and sound speed.
template <class R>
struct State {
    R U0, U1, U2, U3;   // rho, rho*u, rho*v, E
    R u, v, p, E, a;
};

// EulerIdealGasModel::cons_to_prim (model/euler_ideal_gas/euler_ideal_gas.cpp:76-92)
// and prim_total_energy / prim_internal_energy (:32-46).
template <class M>
__device__ __forceinline__ void prims(typename M::R U0, typename M::R U1, typename M::R U2, typename M::R U3,
                                      typename M::R g1, typename M::R& u, typename M::R& v,
                                      typename M::R& p, typename M::R& E)
{
    typedef typename M::R R;
    u = M::div(U1, U0);
    v = M::div(U2, U0);
    const R q2 = u * u + v * v;
    p = g1 * (U3 - R(0.5) * U0 * q2);
    const R e = M::div(p, U0 * g1);
    E = U0 * (R(0.5) * q2 + e);
}

// prim_speed_of_sound (euler_ideal_gas.cpp:60-64), also used by
// calc_wave_speeds_direct_min_max (riemann_hllc.cpp:130-131).
template <class M>
__device__ __forceinline__ typename M::R sound(typename M::R gamma, typename M::R p, typename M::R rho)
{
    return M::sqrt(M::div(gamma * p, rho));
}

// ------------------------------------------------------------ FP32 bulk --
// The FP32 path owes no bit-for-bit contract, so it evaluates the same
// scheme in fewer operations (results agree with the FP64 path to FP32
// rounding):
//  * one reciprocal of rho per state, shared by u, v and the sound speed;
//  * the state's own total energy E where the reference re-derives it from
//    the primitives (rho (q^2/2 + p/(rho (gamma-1))) equals E up to rounding);
//  * rho u and rho v are the conserved momenta themselves in the fluxes;
//  * the limiters with one reciprocal (the ratio and xi(r) folded into one
//    quotient), each difference of neighbours clamped once for the two cells
//    that use it, HLLC's star state with two, the flux of the upwind side only;
//  * multiply-adds written as explicit fmaf.  The build disables contraction,
//    so no other operation is fused and every copy of this code (warm-up and
//    loop body of a sweep) rounds the same way: results do not depend on how
//    the rows are split into work items.
namespace f32 {

__device__ __forceinline__ float fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// the limiter ratio's tolerance clamp (muscl_hancock.cpp:8-11,78-94): |d| is
// raised to 1e-6 under the sign of d, +1e-6 for either zero.  Only momenta
// (ZERO) can differ by -0.  A NaN becomes a number here: see slope().
template <bool ZERO>
__device__ __forceinline__ float clamp_tol(float d)
{
    return __builtin_copysignf(__builtin_fmaxf(__builtin_fabsf(d), 1e-6f), ZERO ? d + 0.0f : d);
}

// Differences b - a of two neighbouring cells, raw and clamped: they serve
// the slopes of both cells.
__device__ __forceinline__ void differences(const float a[4], const float b[4], float d[4], float c[4])
{
    for (int k = 0; k < 4; k++) d[k] = b[k] - a[k];
    c[0] = clamp_tol<false>(d[0]);
    c[1] = clamp_tol<true>(d[1]);
    c[2] = clamp_tol<true>(d[2]);
    c[3] = clamp_tol<false>(d[3]);
}

// u, v, p of a conserved state; ri = 1/rho
__device__ __forceinline__ void prims(float U0, float U1, float U2, float U3, float g1, float& ri, float& u, float& v,
                                      float& p)
{
    ri = rcp(U0);
    u = U1 * ri;
    v = U2 * ri;
    p = g1 * fma(-0.5f, fma(U1, u, U2 * v), U3);
}

__device__ __forceinline__ State<float> make_state(const float U[4], float gamma, float g1)
{
    State<float> s;
    s.U0 = U[0]; s.U1 = U[1]; s.U2 = U[2]; s.U3 = U[3];
    float ri;
    prims(U[0], U[1], U[2], U[3], g1, ri, s.u, s.v, s.p);
    s.E = U[3];
    s.a = __builtin_amdgcn_sqrtf(gamma * s.p * ri);
    return s;
}

// Euler flux normal to the face: X (x-face) or y-face, E = the state's own energy
template <bool X>
__device__ __forceinline__ void flux(float U0, float U1, float U2, float U3, float u, float v, float p, float F[4])
{
    (void)U0;
    if (X) {
        F[0] = U1;
        F[1] = fma(U1, u, p);
        F[2] = U1 * v;
        F[3] = u * (U3 + p);
    } else {
        F[0] = U2;
        F[1] = U2 * u;
        F[2] = fma(U2, v, p);
        F[3] = v * (U3 + p);
    }
}

// HLLC with the Davis wave speeds, Toro's star state rewritten with
// m_K = rho_K (S_K - q_K):  S* = (p_R - p_L + m_L q_L - m_R q_R) / (m_L - m_R),
// U*_K = [m_K, m_K S*, m_K t_K, (S_K - q_K) E_K + (S* - q_K)(m_K S* + p_K)] / (S_K - S*).
// The branch order of the reference: 0 <= S_L full left flux, then the left
// and right star fluxes, 0 >= S_R full right flux, otherwise (NaN) zero.
template <bool X>
__device__ __forceinline__ void hllc(const State<float>& L, const State<float>& Rs, float F[4])
{
    const float qL = X ? L.u : L.v, qR = X ? Rs.u : Rs.v;
    // The reference's std::min / std::max drop a NaN of the right state and
    // keep one of the left: so do these, with the left speeds in `chk`.
    const float aL = qL - L.a, bL = qL + L.a;
    const float S_L = __builtin_fminf(aL, qR - Rs.a);
    const float S_R = __builtin_fmaxf(bL, qR + Rs.a);
    const float mL = L.U0 * (S_L - qL), mR = Rs.U0 * (S_R - qR);
    const float Ss = fma(mL, qL, fma(-mR, qR, Rs.p - L.p)) * rcp(mL - mR);

    // Branch choice of the reference for finite speeds: S_L >= 0 takes the
    // full left flux; otherwise S* >= 0 the left star flux; otherwise the
    // right side, its star flux if S_R >= 0, else the full right flux.  So
    // K = R exactly when S_L < 0 and S* < 0, and the star term's weight
    // S_K (zero for a full flux) is min(S_L, 0) on the left, max(S_R, 0) on
    // the right.  A NaN speed gives the zero flux, as in the reference.
    const bool useR = (S_L < 0.0f) & (Ss < 0.0f);
    const float wL = __builtin_fminf(S_L, 0.0f), wR = __builtin_fmaxf(S_R, 0.0f);
    const float chk = aL + bL + Ss;
    const bool none = !(chk == chk);
    const float dK = useR ? Rs.U0 : L.U0;
    const float U1K = useR ? Rs.U1 : L.U1;
    const float U2K = useR ? Rs.U2 : L.U2;
    const float EK = useR ? Rs.U3 : L.U3;
    const float uK = useR ? Rs.u : L.u;
    const float vK = useR ? Rs.v : L.v;
    const float pK = useR ? Rs.p : L.p;
    const float SK = useR ? S_R : S_L;
    const float mK = useR ? mR : mL;
    const float qK = X ? uK : vK, tK = X ? vK : uK;
    const float UnK = X ? U1K : U2K, UtK = X ? U2K : U1K;

    float FK[4];
    flux<X>(dK, U1K, U2K, EK, uK, vK, pK, FK);
    const float rS = rcp(SK - Ss);
    const float us0 = mK * rS;
    const float us3 = rS * fma(SK - qK, EK, (Ss - qK) * fma(mK, Ss, pK));
    const float w = useR ? wR : wL;
    const bool star = w != 0.0f;   // a full flux never sees the star state (it may not be finite)
    const float d0 = us0 - dK;
    const float dn = fma(us0, Ss, -UnK);
    const float dt = fma(us0, tK, -UtK);
    const float d3 = us3 - EK;
    const float F0 = star ? fma(w, d0, FK[0]) : FK[0];
    const float Fn = star ? fma(w, X ? dn : dt, FK[1]) : FK[1];
    const float Ft = star ? fma(w, X ? dt : dn, FK[2]) : FK[2];
    const float F3 = star ? fma(w, d3, FK[3]) : FK[3];
    F[0] = none ? 0.0f : F0;
    F[1] = none ? 0.0f : Fn;
    F[2] = none ? 0.0f : Ft;
    F[3] = none ? 0.0f : F3;
}

// Limited slope xi(r) * (dl + dr) / 2 with r from the clamped deltas
// (muscl_hancock.cpp:67-206), one reciprocal.  For r > 0 (same signs):
//  MinBee  r <= 1: xi = r              -> (dl+dr)/2 * dlc / drc
//          r >  1: xi = 2/(1+r)        -> (dl+dr) * drc / (drc + dlc)
//  VanLeer xi = 2 min(r, 1)/(1+r)      -> (dl+dr) * m / (dlc + drc), m = dlc or drc, whichever is
//          smaller in magnitude (both have the sign of drc)
// r > 0 where the clamped deltas have one sign; their median with zero is then
// the smaller of them, and zero otherwise.  The product with dl + dr is
// positive in the first case (or dl + dr is zero) and zero or a NaN in the
// others: s is zero there, as it is for a NaN difference in the reference.
template <int LIM>
__device__ __forceinline__ float slope(float dl, float dr, float dlc, float drc)
{
    const float m = __builtin_amdgcn_fmed3f(dlc, drc, 0.0f);
    float num = m, den = dlc + drc;
    if (LIM == 0) {
        const bool le1 = __builtin_fabsf(dlc) <= __builtin_fabsf(drc);   // |r| <= 1
        num = le1 ? 0.5f * m : m;
        den = le1 ? drc : den;
    }
    const float t = (dl + dr) * num;
    return t > 0.0f ? t * rcp(den) : 0.0f;
}

// One direction of MUSCL-Hancock reconstruction of a cell from its
// differences: face states U -+ s/2 and the split half-step predictor
// face += h (F(lo) - F(hi)).
template <int LIM, bool X>
__device__ __forceinline__ void reconstruct(const float uc[4], const float dl[4], const float dr[4], const float cl[4],
                                            const float cr[4], float h, float g1, float lo[4], float hi[4])
{
    for (int k = 0; k < 4; k++) {
        const float s = slope<LIM>(dl[k], dr[k], cl[k], cr[k]);
        lo[k] = fma(-0.5f, s, uc[k]);
        hi[k] = fma(0.5f, s, uc[k]);
    }
    float ri, ul, vl, pl, ur, vr, pr;
    prims(lo[0], lo[1], lo[2], lo[3], g1, ri, ul, vl, pl);
    prims(hi[0], hi[1], hi[2], hi[3], g1, ri, ur, vr, pr);
    float Fl[4], Fr[4];
    flux<X>(lo[0], lo[1], lo[2], lo[3], ul, vl, pl, Fl);
    flux<X>(hi[0], hi[1], hi[2], hi[3], ur, vr, pr, Fr);
    for (int k = 0; k < 4; k++) {
        const float d = Fl[k] - Fr[k];
        lo[k] = fma(h, d, lo[k]);
        hi[k] = fma(h, d, hi[k]);
    }
}
template <int LIM, bool X>
__device__ __forceinline__ void reconstruct(const float um[4], const float uc[4], const float up[4], float h, float g1,
                                            float lo[4], float hi[4])
{
    float dl[4], dr[4], cl[4], cr[4];
    differences(um, uc, dl, cl);
    differences(uc, up, dr, cr);
    reconstruct<LIM, X>(uc, dl, dr, cl, cr, h, g1, lo, hi);
}

// |u| + c and |v| + c of a state (TimeStep's per-cell terms)
__device__ __forceinline__ void wave_speeds(float U0, float U1, float U2, float U3, float gamma, float g1, double& Dx,
                                            double& Dy)
{
    float ri, u, v, p;
    prims(U0, U1, U2, U3, g1, ri, u, v, p);
    const float c = __builtin_amdgcn_sqrtf(gamma * p * ri);
    Dx = (double)(__builtin_fabsf(u) + c);
    Dy = (double)(__builtin_fabsf(v) + c);
}

}  // namespace f32

template <class M>
__device__ __forceinline__ State<typename M::R> make_state(const typename M::R U[4], typename M::R gamma,
                                                           typename M::R g1)
{
    if constexpr (M::fast) {
        return f32::make_state(U, gamma, g1);
    } else {
        State<typename M::R> s;
        s.U0 = U[0]; s.U1 = U[1]; s.U2 = U[2]; s.U3 = U[3];
        prims<M>(U[0], U[1], U[2], U[3], g1, s.u, s.v, s.p, s.E);
        s.a = sound<M>(gamma, s.p, U[0]);
        return s;
    }
}

// cons_flux_x / cons_flux_y (euler_ideal_gas.cpp:113-149) from precomputed
// primitives: [rho u, rho u u + p, rho u v, u (E + p)] and the y mirror.
template <class R, bool X>
__device__ __forceinline__ void flux(R rho, R u, R v, R p, R E, R F[4])
{
    if (X) {
        F[0] = rho * u;
        F[1] = rho * u * u + p;
        F[2] = rho * u * v;
        F[3] = u * (E + p);
    } else {
        F[0] = rho * v;
        F[1] = rho * u * v;
        F[2] = rho * v * v + p;
        F[3] = v * (E + p);
    }
}

// HLLCEulerRiemannSolver::calc_hllc_flux (riemann_hllc.cpp:169-212) with the
// Davis wave speeds (:127-150), S* (:67-97), U*_K (:37-63), F*_K (:153-164).
// NaN or inconsistent states fall through to a zero flux (:207-210).
template <class M, bool X>
__device__ __forceinline__ void hllc(const State<typename M::R>& L, const State<typename M::R>& Rs,
                                     typename M::R F[4])
{
    typedef typename M::R R;
    if constexpr (M::fast) {
        f32::hllc<X>(L, Rs, F);
        return;
    }
    const R qL = X ? L.u : L.v, qR = X ? Rs.u : Rs.v;
    const R S_L = smin(qL - L.a, qR - Rs.a);
    const R S_R = smax(qL + L.a, qR + Rs.a);
    const R num = Rs.p - L.p + L.U0 * qL * (S_L - qL) - Rs.U0 * qR * (S_R - qR);
    const R den = L.U0 * (S_L - qL) - Rs.U0 * (S_R - qR);
    const R Ss = M::div(num, den);

    const bool c1 = R(0) <= S_L;
    const bool c2 = (S_L <= R(0)) && (R(0) <= Ss);
    const bool c3 = (Ss <= R(0)) && (R(0) <= S_R);
    const bool c4 = R(0) >= S_R;
    const bool useR = !c1 && !c2 && c3;   // F*_R branch; otherwise the star state of L

    // the side whose star state is needed
    const R dK = useR ? Rs.U0 : L.U0;
    const R uK = useR ? Rs.u : L.u;
    const R vK = useR ? Rs.v : L.v;
    const R pK = useR ? Rs.p : L.p;
    const R EK = useR ? Rs.E : L.E;
    const R SK = useR ? S_R : S_L;
    const R qK = X ? uK : vK;
    const R tK = X ? vK : uK;
    const R coef = dK * M::div(SK - qK, SK - Ss);
    const R us0 = coef;
    const R usn = coef * Ss;
    const R ust = coef * tK;
    const R us3 = coef * (M::div(EK, dK) + (Ss - qK) * (Ss + M::div(pK, dK * (SK - qK))));

    R FL[4], FR[4];
    flux<R, X>(L.U0, L.u, L.v, L.p, L.E, FL);
    flux<R, X>(Rs.U0, Rs.u, Rs.v, Rs.p, Rs.E, FR);
    const R K0 = useR ? Rs.U0 : L.U0;
    const R K1 = useR ? Rs.U1 : L.U1;
    const R K2 = useR ? Rs.U2 : L.U2;
    const R K3 = useR ? Rs.U3 : L.U3;
    R FK[4];
    for (int i = 0; i < 4; i++) FK[i] = useR ? FR[i] : FL[i];
    R Fs[4];
    Fs[0] = FK[0] + SK * (us0 - K0);
    Fs[1] = FK[1] + SK * ((X ? usn : ust) - K1);
    Fs[2] = FK[2] + SK * ((X ? ust : usn) - K2);
    Fs[3] = FK[3] + SK * (us3 - K3);

    for (int i = 0; i < 4; i++) {
        R f = R(0);
        if (c1) f = FL[i];
        else if (c2 || c3) f = Fs[i];
        else if (c4) f = FR[i];
        F[i] = f;
    }
}

// Tolerance clamp of the limiter ratio (scheme/muscl_hancock/muscl_hancock.cpp:8-11,78-94).
template <class M>
__device__ __forceinline__ typename M::R clamp_delta(typename M::R d)
{
    typedef typename M::R R;
    const R tol = R(M::tol);
    if (M::fabs(d) <= tol) return (d == R(0)) ? tol : ((d > R(0)) ? tol : -tol);
    return d;
}

// MinBeeLimiter::operator() (scheme/limiter/minbee/minbee.cpp:29-38) and
// VanLeerLimiter::operator() (scheme/limiter/vanleer/vanleer.cpp:29-36) with
// omega=0, beta=1 (parser.cpp:231,233); xi_right = 2/(1+r) (limiter.cpp:48-53),
// whose denominator guard never triggers on the evaluated branches.
template <class M, int LIM>
__device__ __forceinline__ typename M::R limiter(typename M::R r)
{
    typedef typename M::R R;
    if (LIM == 0) {
        const R x = M::div(R(2), R(1) + r);
        return (r <= R(0)) ? R(0) : ((r <= R(1)) ? r : ((x < R(1)) ? x : R(1)));
    } else {
        // min(2r/(1+r), 2/(1+r)) with one division; r = +inf gives inf/inf = NaN
        // exactly as std::min(NaN, 0) does in the reference.
        const R inf = __builtin_huge_val();
        const R num = (r < R(1)) ? R(2) * r : ((r == inf) ? inf : R(2));
        const R x = M::div(num, R(1) + r);
        return (r <= R(0)) ? R(0) : x;
    }
}

// Limited slope of one conserved variable (muscl_hancock.cpp:137-206):
// xi(r) * (0.5*(1+omega)*dl + 0.5*(1-omega)*dr) with unclamped deltas.
template <class M, int LIM>
__device__ __forceinline__ typename M::R slope(typename M::R um, typename M::R uc, typename M::R up)
{
    typedef typename M::R R;
    const R dl = uc - um;
    const R dr = up - uc;
    const R r = M::div(clamp_delta<M>(dl), clamp_delta<M>(dr));
    return limiter<M, LIM>(r) * (R(0.5) * dl + R(0.5) * dr);
}

// One direction of MUSCL-Hancock reconstruction for one cell: boundary
// extrapolation (muscl_hancock.cpp:209-240) and the direction-split half-step
// predictor (:243-281): lo/hi are the face states (L,R) or (B,T).
template <class M, int LIM, bool X>
__device__ __forceinline__ void reconstruct(const typename M::R um[4], const typename M::R uc[4],
                                            const typename M::R up[4], typename M::R h, typename M::R g1,
                                            typename M::R lo[4], typename M::R hi[4])
{
    typedef typename M::R R;
    if constexpr (M::fast) {
        f32::reconstruct<LIM, X>(um, uc, up, h, g1, lo, hi);
        return;
    }
    for (int k = 0; k < 4; k++) {
        const R s = slope<M, LIM>(um[k], uc[k], up[k]);
        lo[k] = uc[k] - R(0.5) * s;
        hi[k] = uc[k] + R(0.5) * s;
    }
    R ul, vl, pl, El, ur, vr, pr, Er;
    prims<M>(lo[0], lo[1], lo[2], lo[3], g1, ul, vl, pl, El);
    prims<M>(hi[0], hi[1], hi[2], hi[3], g1, ur, vr, pr, Er);
    R Fl[4], Fr[4];
    flux<R, X>(lo[0], ul, vl, pl, El, Fl);
    flux<R, X>(hi[0], ur, vr, pr, Er, Fr);
    for (int k = 0; k < 4; k++) {
        const R d = Fl[k] - Fr[k];
        lo[k] += h * d;
        hi[k] += h * d;
    }
}

// ------------------------------------------------- FP64 within range --
// The same FP64 results, bit for bit, for states whose magnitudes keep every
// quotient and root away from the ends of the exponent range.
//
// IEEE division compiles to v_div_scale (twice), a reciprocal with two Newton
// steps, the quotient with one residual correction, v_div_fmas and
// v_div_fixup: 11 instructions and a quarter-rate reciprocal.  Where neither
// operand, the reciprocal, the quotient nor the residual leaves the normal
// range, the scales return their operands, v_div_fmas is the plain
// multiply-add and the fix-up changes nothing, so the eight operations in
// between give the same bits -- and the reciprocal half of them is shared by
// all quotients of one denominator (u, v and the sound speed of a state, the
// star state's E/rho).  The square root drops its scaling the same way.
//
// What can differ is caught by masks that every function adds lanes to:
//  * rows of conserved values are checked by out_of_range(): density and
//    energy within [2^-60, 2^40], momenta zero or at least 2^-800;
//  * face densities and pressures (>= 2^-60) and the numerator of S* (zero or
//    at least 2^-800) are checked where they arise; a transverse momentum that is zero on one
//    side of a cell only could become a product of two tiny values, and
//    counts as out of range;
//  * a quotient by zero, an overflow or a NaN makes the new state's wave
//    speed NaN, which the sweeps test.
// With these bounds, gamma - 1 in [2^-10, 2^10] and h = dt/(2 dx) in [2^-100,
// 2^20], a non-zero slope-limited momentum is at least 2^-858 (the limiter's
// clamp gives xi = 1 wherever both differences are below 1e-6, and any other
// slope is at least 2^-84), after the predictor at least 2^-912, and densities
// stay below 2^64: numerators above 2^-968 and quotients above 2^-1022, where
// the residual a - b q is exact.  A sweep that finds a lane out of range
// leaves the row, and the rest of its item, to the general code below it; one
// that finds its first rows out of range does so before any arithmetic.  Such
// states (units far from 1) then cost a second request of those rows, us per
// step by the general code alone / found after the first face / found at once:
// Van Leer 50^2 11.8 / 14.2 / 12.9, 300^2 17.1 / 19.5 / 18.2, 2048^2 215 / 218 /
// 215, Godunov 400^2 12.1 / 13.4 / 13.0, unstructured 367 500 cells 25.9 / 38.6 /
// 25.0.
//
// In assembly, one row of k_muscl (60 cells) went from 1 397 (MinBee) and
// 1 429 (Van Leer) to 970 and 975 VALU instructions, 60 of them quarter-rate
// to 36 (general rows now 1 371 and 1 401).  8192^2 Van Leer: 3.13 -> 2.41 ms per step, the 8 x
// 1024^2 channel 0.440 -> 0.379, Godunov 400^2 0.0258 -> 0.0248.
namespace q64 {

__device__ __forceinline__ double fma(double a, double b, double c) { return __builtin_fma(a, b, c); }

// The bounds and the limiter's constants, in vector registers: as literals
// they would sit in scalar ones, and a row loop short of those moves others to
// and from vector lanes (up to 65 instructions a row).
struct Limits {
    double low = 0x1p-60, high = 0x1p40, tiny = 0x1p-800, tol = 1e-6, quarter = 0.25;
    __device__ __forceinline__ Limits()
    {
        asm volatile("" : "+v"(low), "+v"(high), "+v"(tiny), "+v"(tol), "+v"(quarter));
    }
};

typedef unsigned long long mask;   // lanes, as __ballot gives them

// 1/b by the division's own steps
__device__ __forceinline__ double rcp(double b)
{
    const double r0 = __builtin_amdgcn_rcp(b);
    const double r1 = fma(r0, fma(-b, r0, 1.0), r0);
    return fma(r1, fma(-b, r1, 1.0), r1);
}
// a/b from y = rcp(b).  For b > 0 a zero numerator keeps its sign: the
// residual is taken as b q - a, so that the correction adds a zero of q's sign.
__device__ __forceinline__ double div_pos(double a, double b, double y)
{
    const double q = a * y;
    return fma(-fma(b, q, -a), y, q);
}
// the same for b < 0 (also for any b and a != 0)
__device__ __forceinline__ double div_neg(double a, double b, double y)
{
    const double q = a * y;
    return fma(fma(-b, q, a), y, q);
}
// The compiler's own steps for the correctly rounded square root, 0 < x in range.
__device__ __forceinline__ double sqrt(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    const double g0 = x * y, h0 = 0.5 * y;
    const double r0 = fma(-h0, g0, 0.5);
    const double h1 = fma(h0, r0, h0), g1 = fma(g0, r0, g0);
    const double g2 = fma(fma(-g1, g1, x), h1, g1);
    return fma(fma(-g2, g2, x), h1, g2);
}

// Lanes whose conserved state is out of range.
__device__ __forceinline__ mask out_of_range(const double U[4], const Limits& c)
{
    return __ballot(!(U[0] >= c.low)) | __ballot(!(U[0] <= c.high)) | __ballot(!(U[3] >= c.low)) |
           __ballot(!(U[3] <= c.high)) | (__ballot(U[1] != 0.0) & __ballot(__builtin_fabs(U[1]) < c.tiny)) |
           (__ballot(U[2] != 0.0) & __ballot(__builtin_fabs(U[2]) < c.tiny));
}
// Constants of a launch and the half steps of an item.
__device__ __forceinline__ bool constants_in_range(double gamma, double g1)
{
    return g1 >= 0x1p-10 && g1 <= 0x1p10 && gamma > 0.0;
}
__device__ __forceinline__ bool half_step_in_range(double h) { return h >= 0x1p-100 && h <= 0x1p20; }

struct State {
    double U0, U1, U2, U3;
    double u, v, p, E, a;
    double y;   // rcp(U0)
};

// Primitives and total energy; ig1 = 1/(gamma - 1) starts the reciprocal of
// rho (gamma - 1) from that of rho, one Newton step short of it.
__device__ __forceinline__ void prims(double U0, double U1, double U2, double U3, double g1, double ig1, double& y,
                                      double& u, double& v, double& p, double& E, mask& bad, const Limits& lim)
{
    y = rcp(U0);
    u = div_pos(U1, U0, y);
    v = div_pos(U2, U0, y);
    const double q2 = u * u + v * v;
    p = g1 * fma(-0.5, U0 * q2, U3);   // halving is exact: the reference's U3 - 0.5 rho q2
    const double c = U0 * g1;
    const double y0 = y * ig1;
    const double yc = fma(y0, fma(-c, y0, 1.0), y0);
    E = U0 * fma(0.5, q2, div_pos(p, c, yc));
    bad |= __ballot(!(U0 >= lim.low)) | __ballot(!(p >= lim.low));
}

__device__ __forceinline__ State make_state(const double U[4], double gamma, double g1, double ig1, mask& bad,
                                            const Limits& lim)
{
    State s;
    s.U0 = U[0]; s.U1 = U[1]; s.U2 = U[2]; s.U3 = U[3];
    prims(U[0], U[1], U[2], U[3], g1, ig1, s.y, s.u, s.v, s.p, s.E, bad, lim);
    s.a = sqrt(div_pos(gamma * s.p, s.U0, s.y));
    return s;
}

// The limiter's clamped difference: |d| raised to 1e-6 under the sign of d,
// +1e-6 for either zero.  Only momenta (ZERO) can differ by -0.
template <bool ZERO>
__device__ __forceinline__ double clamp_delta(double d, const Limits& lim)
{
    return __builtin_copysign(__builtin_fmax(__builtin_fabs(d), lim.tol), ZERO ? d + 0.0 : d);
}

// Differences b - a of two neighbouring cells, raw and clamped.
__device__ __forceinline__ void differences(const double a[4], const double b[4], double d[4], double c[4],
                                            const Limits& lim)
{
    for (int k = 0; k < 4; k++) d[k] = b[k] - a[k];
    c[0] = clamp_delta<false>(d[0], lim);
    c[1] = clamp_delta<true>(d[1], lim);
    c[2] = clamp_delta<true>(d[2], lim);
    c[3] = clamp_delta<false>(d[3], lim);
}

// Twice the limited slope's numerator: xi(r) (dl + dr), from the raw and the
// clamped differences.  r is finite and non-zero; for r > 1, 2/(1+r) <= 1.
template <int LIM>
__device__ __forceinline__ double limited_sum(double dl, double dr, double cl, double cr)
{
    const double r = div_neg(cl, cr, rcp(cr));
    const double b = 1.0 + r;
    const double num = (LIM != 0 && r < 1.0) ? 2.0 * r : 2.0;
    const double x = div_pos(num, b, rcp(b));
    const double xi = (LIM == 0 && r <= 1.0) ? r : x;
    return (r <= 0.0 ? 0.0 : xi) * (dl + dr);
}

// Face states of a cell from its differences: U -+ 0.25 xi (dl + dr) (the
// reference's U -+ 0.5 xi (0.5 dl + 0.5 dr): every factor 0.5 is exact), then
// the split half-step predictor.
template <int LIM, bool X>
__device__ __forceinline__ void reconstruct(const double uc[4], const double dl[4], const double dr[4],
                                            const double cl[4], const double cr[4], double h, double g1, double ig1,
                                            double lo[4], double hi[4], mask& bad, const Limits& lim)
{
    for (int k = 0; k < 4; k++) {
        const double w = limited_sum<LIM>(dl[k], dr[k], cl[k], cr[k]);
        lo[k] = fma(-lim.quarter, w, uc[k]);
        hi[k] = fma(lim.quarter, w, uc[k]);
    }
    constexpr int T = X ? 2 : 1;   // the transverse momentum
    bad |= __ballot(lo[T] == 0.0) ^ __ballot(hi[T] == 0.0);
    double y, ul, vl, pl, El, ur, vr, pr, Er;
    prims(lo[0], lo[1], lo[2], lo[3], g1, ig1, y, ul, vl, pl, El, bad, lim);
    prims(hi[0], hi[1], hi[2], hi[3], g1, ig1, y, ur, vr, pr, Er, bad, lim);
    double Fl[4], Fr[4];
    flux<double, X>(lo[0], ul, vl, pl, El, Fl);
    flux<double, X>(hi[0], ur, vr, pr, Er, Fr);
    for (int k = 0; k < 4; k++) {
        const double d = Fl[k] - Fr[k];
        lo[k] += h * d;
        hi[k] += h * d;
    }
}

// The general hllc() for finite wave speeds: the side K is the right one
// exactly when S_L < 0 and S* < 0, and only its flux and star state are
// evaluated; the star flux holds unless the whole fan lies on K's far side.
template <bool X>
__device__ __forceinline__ void hllc(const State& L, const State& Rs, double F[4], mask& bad, const Limits& lim)
{
    const double qL = X ? L.u : L.v, qR = X ? Rs.u : Rs.v;
    const double S_L = __builtin_fmin(qL - L.a, qR - Rs.a);
    const double S_R = __builtin_fmax(qL + L.a, qR + Rs.a);
    const double num = Rs.p - L.p + L.U0 * qL * (S_L - qL) - Rs.U0 * qR * (S_R - qR);
    const double den = L.U0 * (S_L - qL) - Rs.U0 * (S_R - qR);
    bad |= __ballot(num != 0.0) & __ballot(__builtin_fabs(num) < lim.tiny);
    const double Ss = div_neg(num, den, rcp(den));

    const bool useR = (S_L < 0.0) & (Ss < 0.0);
    const double dK = useR ? Rs.U0 : L.U0;
    const double uK = useR ? Rs.u : L.u;
    const double vK = useR ? Rs.v : L.v;
    const double pK = useR ? Rs.p : L.p;
    const double EK = useR ? Rs.E : L.E;
    const double SK = useR ? S_R : S_L;
    const double yK = useR ? Rs.y : L.y;
    const double K1 = useR ? Rs.U1 : L.U1;
    const double K2 = useR ? Rs.U2 : L.U2;
    const double K3 = useR ? Rs.U3 : L.U3;
    const double qK = X ? uK : vK, tK = X ? vK : uK;
    double FK[4];
    flux<double, X>(dK, uK, vK, pK, EK, FK);
    const double sq = SK - qK, ss = SK - Ss, D = dK * sq;
    const double coef = dK * div_neg(sq, ss, rcp(ss));
    const double us3 = coef * (div_pos(EK, dK, yK) + (Ss - qK) * (Ss + div_neg(pK, D, rcp(D))));
    const bool star = useR ? (0.0 <= S_R) : (S_L < 0.0);
    const double usn = coef * Ss, ust = coef * tK;
    const double d[4] = {coef - dK, (X ? usn : ust) - K1, (X ? ust : usn) - K2, us3 - K3};
    for (int i = 0; i < 4; i++) F[i] = star ? FK[i] + SK * d[i] : FK[i];
}

// wave_speeds() of a new state; its own range is checked here (a pressure of
// zero or below makes the speed NaN, which the caller tests).
__device__ __forceinline__ void wave_speeds(const double U[4], double gamma, double g1, double& Dx, double& Dy,
                                            mask& bad, const Limits& lim)
{
    const double y = rcp(U[0]);
    const double u = div_pos(U[1], U[0], y), v = div_pos(U[2], U[0], y);
    const double p = g1 * fma(-0.5, U[0] * (u * u + v * v), U[3]);
    const double c = sqrt(div_pos(gamma * p, U[0], y));
    Dx = __builtin_fabs(u) + c;
    Dy = __builtin_fabs(v) + c;
    bad |= __ballot(!(U[0] >= lim.low)) | __ballot(!(U[3] >= lim.low)) | __ballot(!(Dx == Dx));
}

}  // namespace q64

// calculate_spatial_update (muscl_hancock.cpp:364-371, godunov.cpp:97-111)
// and the forward Euler step (dt*L)+U (forward_euler.cpp:27-28): the
// reference's order in FP64, multiply-adds in FP32.
template <class M>
__device__ __forceinline__ void update_cell(typename M::R rdx, typename M::R rdy, typename M::R dt,
                                            const typename M::R Fw[4], const typename M::R Fe[4],
                                            const typename M::R Gs[4], const typename M::R Gn[4],
                                            const typename M::R U[4], typename M::R L[4], typename M::R Un[4])
{
    for (int k = 0; k < 4; k++) {
        if constexpr (M::fast) {
            L[k] = f32::fma(rdx, Fw[k] - Fe[k], rdy * (Gs[k] - Gn[k]));
            Un[k] = f32::fma(dt, L[k], U[k]);
        } else {
            L[k] = rdx * (Fw[k] - Fe[k]) + rdy * (Gs[k] - Gn[k]);
            Un[k] = dt * L[k] + U[k];
        }
    }
}

// Bits of a non-negative double; their unsigned order is the numeric order,
// which lets wave-speed maxima use 64-bit integer atomics.
__device__ __forceinline__ unsigned long long dbits(double x) { return (unsigned long long)__double_as_longlong(x); }
__device__ __forceinline__ double bitsd(unsigned long long b) { return __longlong_as_double((long long)b); }

// Largest |u|+c and |v|+c of a conserved state (the per-cell terms of
// TimeStep::operator(), timestep.cpp:42-52); NaN terms are skipped by the caller.
template <class M>
__device__ __forceinline__ void wave_speeds(typename M::R U0, typename M::R U1, typename M::R U2,
                                            typename M::R U3, typename M::R gamma, typename M::R g1,
                                            double& Dx, double& Dy)
{
    typedef typename M::R R;
    if constexpr (M::fast) {
        f32::wave_speeds(U0, U1, U2, U3, gamma, g1, Dx, Dy);
        return;
    }
    const R u = M::div(U1, U0);
    const R v = M::div(U2, U0);
    const R p = g1 * (U3 - R(0.5) * U0 * (u * u + v * v));
    const R c = sound<M>(gamma, p, U0);
    Dx = (double)(M::fabs(u) + c);
    Dy = (double)(M::fabs(v) + c);
}

__device__ __forceinline__ double dmax_nan(double acc, double x) { return (x > acc) ? x : acc; }

// Reduction of a per-lane value over the wave by DPP: within rows of 16 lanes
// by shifts, then row ends broadcast into the next rows; lane 63 ends with the
// whole wave's, which every lane gets (a scalar).  About 30 instructions
// without an LDS round trip, where six bpermute shuffles of a double wait for
// twelve.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_f64(double x)   // the partner's x, or x where there is none
{
    const long long b = __double_as_longlong(x);
    const int lo = (int)(b & 0xffffffffll), hi = (int)(b >> 32);
    const int l2 = __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xf, false);
    const int h2 = __builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xf, false);
    return __longlong_as_double(((long long)h2 << 32) | (unsigned int)l2);
}
template <class F>
__device__ __forceinline__ double wave_prefix(double x, F pick)   // over lanes 0..lane
{
    x = pick(x, dpp_f64<0x111, 0xf>(x));   // row_shr:1, 2, 4, 8
    x = pick(x, dpp_f64<0x112, 0xf>(x));
    x = pick(x, dpp_f64<0x114, 0xf>(x));
    x = pick(x, dpp_f64<0x118, 0xf>(x));
    x = pick(x, dpp_f64<0x142, 0xa>(x));   // row_bcast:15 into rows 1 and 3
    x = pick(x, dpp_f64<0x143, 0xc>(x));   // row_bcast:31 into rows 2 and 3
    return x;
}
__device__ __forceinline__ double lane_value(double x, int lane)   // the same for every lane
{
    const long long b = __double_as_longlong(x);
    const unsigned lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), lane);
    const unsigned hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <class F>
__device__ __forceinline__ double wave_reduce(double x, F pick)
{
    return lane_value(wave_prefix(x, pick), 63);
}

// Maximum / minimum over the wave (NaN-free inputs; every lane calls).
__device__ __forceinline__ double wave_max(double x)
{
    return wave_reduce(x, [](double a, double b) { return (b > a) ? b : a; });
}
__device__ __forceinline__ double wave_min(double x)
{
    return wave_reduce(x, [](double a, double b) { return (b < a) ? b : a; });
}

// The step and predictor dt of a block from the device partial maxima
// (TimeStep::operator(), timestep.cpp:29-68).  For a block the minimum of
// dx/(|u|+c) over its cells equals dx / max(|u|+c): correctly rounded
// division is monotone in the divisor.  A block whose terms were all NaN has
// max 0 and contributes dx/0 = inf, which the 1e16 start value absorbs.
__device__ __forceinline__ double cfl_eff(double cfl, long long call)
{
    return (call <= 10) ? 0.2 * cfl : cfl;   // timestep.cpp:60-65,72,75
}

// Step dt and speculative predictor dt of a block: every block of the
// problem at U^n.  The reference's compat predictor dt (simulation.cpp:106-110
// with muscl_hancock.cpp:246) sees the blocks before this one at U^{n+1}; the
// fix-up launches below compute it and recompute a block whenever the two
// differ.  In uniform mode (or for Godunov, which has no predictor) the
// predictor dt is the step dt.
template <class R>
__device__ __forceinline__ void step_dts(const HfStepArgs<R>& a, const HfBlockDev& bd, bool muscl, double& dt_step,
                                         double& dt_pred, long long& kstep, long long& kpred)
{
    // Lane l takes blocks first+l, first+l+64, ...: the per-block loads and
    // divisions run side by side instead of as one dependent chain, then the
    // minima are reduced over the wave.  A minimum of non-NaN values does not
    // depend on the order, so the results equal the sequential loop's.  Every
    // lane of the wave calls this (wave-uniform arguments).
    const HfProbDev pr = a.probs[bd.problem];
    kstep = (long long)a.calls[bd.problem] - (a.mirrored ? 0 : pr.cps) + 1;
    kpred = kstep + 1 + bd.lb;
    // A lane takes one slot of a block: the quotient by the largest of a
    // block's maxima is the least of the quotients by each.
    double dtx = 1e16, dty = 1e16;
    const int n = pr.nb * a.ways;
    for (int e = (int)(threadIdx.x & 63); e < n; e += 64) {
        const int c = pr.first + e / a.ways;
        const int64_t s = HF_MAX_SLOT(pr.first, e, a.ways, a.way_stride);
        const double cdx = a.blocks[c].dx, cdy = a.blocks[c].dy;
        const double gx = bitsd(a.gmax[2 * c]), gy = bitsd(a.gmax[2 * c + 1]);
        const double ox = smax(bitsd(a.imax_old[s]), gx), oy = smax(bitsd(a.imax_old[s + 1]), gy);
        dtx = smin(dtx, cdx / ox);
        dty = smin(dty, cdy / oy);
    }
    dtx = wave_min(dtx);
    dty = wave_min(dty);
    dt_step = cfl_eff(a.cfl, kstep) * smin(dtx, dty);
    dt_pred = (muscl && a.dt_mode == 0) ? cfl_eff(a.cfl, kpred) * smin(dtx, dty) : dt_step;
}

// ------------------------------------------------------ fix-up planning --
// The compat predictor dt of block l of a problem is cfl_eff(k_l) times
//     min(1e16, min over c < l of pre_c, min over c >= l of old_c)
// with old_c = min(dx_c / max(old x maxima, x ghosts), dy_c / max(old y
// maxima, y ghosts)) (block c at U^n) and pre_c the same with block c's final
// U^{n+1} maxima: a minimum over one set of non-NaN terms, so any grouping
// gives the reference's bits (step_dts takes the x and y minima apart and
// then their minimum, the same set).  The speculative dt of the main list is
// cfl_eff(k_l) * min(1e16, min over all c of old_c); the step dt is
// cfl_eff(k_step) times the same minimum.

// min(dx_c / mx, dy_c / my) for the given maxima bit patterns of block c's
// interior and its ghosts'
template <class R>
__device__ __forceinline__ double term_new(const HfStepArgs<R>& a, int c, unsigned long long mx, unsigned long long my)
{
    const double cdx = a.blocks[c].dx, cdy = a.blocks[c].dy;
    const double gx = bitsd(a.gmax[2 * c]), gy = bitsd(a.gmax[2 * c + 1]);
    return smin(cdx / smax(bitsd(mx), gx), cdy / smax(bitsd(my), gy));
}

// The same from the block's slots in a maxima array.  All slots are requested
// at once (of fewer than HF_MAX_BLOCK_SLOTS, some twice): one round trip to the
// caches, where a loop over the slots took one for each, and the guess and check
// launches' plans wait for little else.  Shortest guess / check launch, us, by
// such a loop with every plan reading its own terms and scanning through LDS,
// and now: 8 x 97^2 channel 7.0 / 9.4, 4.4 / 5.2; 8 x 1024^2 10.1 / 10.4, 5.6 /
// 6.4; 16 channels of 8 x 97^2 in one context 38 / 62, 27 / 40.
template <class R>
__device__ __forceinline__ double term_slots(const HfStepArgs<R>& a, int c, const unsigned long long* m)
{
    typedef unsigned long long pair __attribute__((ext_vector_type(2)));
    const pair* p = (const pair*)(m + HF_MAX_SLOT(c, 0, a.ways, a.way_stride));
    pair v = p[0];
    if (a.ways > 1) {
        pair s[HF_MAX_BLOCK_SLOTS];
        for (int w = 1; w < HF_MAX_BLOCK_SLOTS; w++) s[w] = p[(w & (a.ways - 1)) * (a.way_stride / 2)];
        for (int w = 1; w < HF_MAX_BLOCK_SLOTS; w++) {
            v.x = s[w].x > v.x ? s[w].x : v.x;
            v.y = s[w].y > v.y ? s[w].y : v.y;
        }
    }
    return term_new(a, c, v.x, v.y);
}

template <class R>
__device__ __forceinline__ double term_old(const HfStepArgs<R>& a, int c)
{
    return term_slots(a, c, a.imax_old);
}

// Which maxima are final for pre_c:
//  PRE_MAIN  - the main launch's (at the start of the guess launch nothing has
//              been recomputed);
//  PRE_GUESS - the guess launch's where it recomputed the block, else the
//              main launch's (at the start of the check launch);
//  PRE_CHECK - in the check launch, also the blocks it has recomputed so far:
//              written by other waves of the same launch, so the check
//              launch's slot is read with coherent_read.
enum { PRE_MAIN = 0, PRE_GUESS = 1, PRE_CHECK = 2 };

// A word that other waves of the same launch update with device-scope
// atomics, read with a device-scope atomic read-modify-write that changes
// nothing: it is performed where those atomics are, so it sees every one of
// them that has completed.  A plain atomic load may be served by the reading
// XCD's own L2 from a line cached before those updates.
__device__ __forceinline__ unsigned coherent_read(uint32_t* p)
{
    return __hip_atomic_fetch_or(p, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long coherent_read(unsigned long long* p)
{
    return __hip_atomic_fetch_or(p, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <class R, int SRC>
__device__ __forceinline__ double term_pre(const HfStepArgs<R>& a, int nb_all, int c)
{
    unsigned long long* fix1 = a.imax_fix + HF_MAX_SLOT(nb_all + c, 0, a.ways, a.way_stride);
    if (SRC == PRE_CHECK) {
        const bool f2 = coherent_read(&a.fixed[nb_all + c]) != 0u;
        const unsigned long long x2 = coherent_read(&fix1[0]);
        const unsigned long long y2 = coherent_read(&fix1[1]);
        if (f2) return term_new(a, c, x2, y2);
    }
    return term_slots(a, c, (SRC != PRE_MAIN && a.fixed[c]) ? a.imax_fix : a.imax_new);
}

// Inclusive minimum over lanes 0..lane (scan_lo) or lane..63 (scan_hi).
__device__ __forceinline__ double scan_min_lo(double x)
{
    return wave_prefix(x, [](double a, double b) { return (b < a) ? b : a; });
}
__device__ __forceinline__ double scan_min_hi(double x)
{
    // within rows of 16 lanes, then the minima of the rows above (their first lanes')
    x = smin(x, dpp_f64<0x101, 0xf>(x));   // row_shl:1, 2, 4, 8
    x = smin(x, dpp_f64<0x102, 0xf>(x));
    x = smin(x, dpp_f64<0x104, 0xf>(x));
    x = smin(x, dpp_f64<0x108, 0xf>(x));
    const double r3 = lane_value(x, 48), r2 = smin(lane_value(x, 32), r3), r1 = smin(lane_value(x, 16), r2);
    const int row = (int)(threadIdx.x & 63) >> 4;
    const double above = row == 0 ? r1 : row == 1 ? r2 : r3;
    return row == 3 ? x : smin(x, above);
}

// The fix-up plan of one problem from maxima written by earlier launches
// (plain loads), in one pass over its blocks, 64 at a time (lane <-> block):
// suffix minima of old_c and prefix minima of pre_c give every block's
// predictor dt at once.
//  GUESS (SRC = PRE_MAIN): returns the first block l >= 1 the main list got
//    wrong (skipped, or its speculative dt differs from the exact one) and in
//    m that block's minimum; nb if none.  The guess launch computes every
//    block from there on with cfl_eff(k_l) * min(1e16, m), the exact dt in
//    case no block it recomputes sets a new minimum, and needs to touch
//    block l >= first only if that differs from its speculative dt or the
//    main list skipped it.
//  CHECK (SRC = PRE_GUESS, m = the guess minimum): returns the first block
//    l >= 1 whose computed dt is not the exact one, nb if none, and records
//    the next step's skip verdicts (exact != speculative) of the blocks up to
//    it when `record`.
// O: the problem's speculative minimum min(1e16, min over c of old_c).
// first64: plan_terms(), which the caller's O needs too.
struct PlanTerms {
    double o, n;   // old_c and pre_c by the main launch's maxima; infinite past the last block
};
// The terms of this lane's block of the problem's first 64.
template <class R>
__device__ __forceinline__ PlanTerms plan_terms(const HfStepArgs<R>& a, const HfProbDev& pr, int nb_all)
{
    const int lane = threadIdx.x & 63;
    const double inf = __builtin_huge_val();
    PlanTerms t = {inf, inf};
    if (lane < pr.nb) {
        t.o = term_old(a, pr.first + lane);
        t.n = term_pre<R, PRE_MAIN>(a, nb_all, pr.first + lane);
    }
    return t;
}
template <class R, int SRC>
__device__ int plan_scan(const HfStepArgs<R>& a, const HfProbDev& pr, int nb_all, long long kstep, double O,
                         const PlanTerms& first64, double& m, bool record)
{
    const int lane = threadIdx.x & 63;
    const int nb = pr.nb;
    const double inf = __builtin_huge_val();
    double carry = inf;   // minimum of pre_c over the chunks before this one
    for (int c0 = 0; c0 < nb; c0 += 64) {
        const int c = c0 + lane;
        const bool in = c < nb;
        const int b = pr.first + (in ? c : 0);
        double o = first64.o, n = first64.n;
        if (c0 > 0) {
            o = n = inf;
            if (in) {
                o = term_old(a, b);
                n = term_pre<R, SRC>(a, nb_all, b);
            }
        } else if (SRC == PRE_GUESS && in && a.fixed[b]) {
            n = term_slots(a, b, a.imax_fix);
        }
        double tail = inf;   // minimum of old_c after this chunk
        if (c0 + 64 < nb) {
            for (int t = c0 + 64 + lane; t < nb; t += 64) tail = smin(tail, term_old(a, pr.first + t));
            tail = wave_min(tail);
        }
        double pre = dpp_f64<0x138, 0xf>(scan_min_lo(n));   // wave_shr:1
        pre = (lane == 0 || pre > carry) ? carry : pre;
        double suf = scan_min_hi(o);
        suf = (tail < suf) ? tail : suf;
        const double e = (pre < suf) ? pre : suf;
        const double cf = cfl_eff(a.cfl, kstep + 1 + c);
        const double exact = cf * smin(1e16, e);
        const double spec = cf * smin(1e16, O);
        bool busy;
        if (SRC == PRE_MAIN) {
            busy = in && c >= 1 && (a.skip[b] != 0u || spec != exact);
        } else {
            const bool g = a.fixed[b] != 0u;
            const double used = g ? cf * smin(1e16, m) : spec;
            busy = in && c >= 1 && ((!g && a.skip[b] != 0u) || used != exact);
        }
        const unsigned long long bal = __ballot(busy);
        const int first = bal ? __builtin_ctzll(bal) : 64;
        if (SRC == PRE_GUESS && record && in && c >= 1 && lane <= first) a.skip_next[b] = spec != exact ? 1u : 0u;
        if (bal) {
            if (SRC != PRE_GUESS) m = __shfl(e, first, 64);
            return c0 + first;
        }
        if (c0 + 64 < nb) carry = smin(carry, wave_min(n));
    }
    return nb;
}

// The check launch's verdict on block lb of problem p once every block
// before it is final (the launch has completed every earlier round): the
// step dt, the exact predictor dt and whether the block must be (re)computed
// -- its dt so far (the guess launch's, with guess minimum mg, or the main
// list's speculative one) is not the exact one.  Records the next step's skip
// verdict.
template <class R>
__device__ __forceinline__ bool check_verdict(const HfStepArgs<R>& a, int p, const HfProbDev& pr, int nb_all, int lb,
                                              double mg, double& dt_step, double& dt_pred, long long& kstep,
                                              long long& kpred)
{
    const int block = pr.first + lb;
    kstep = (long long)a.calls[p] - pr.cps + 1;
    kpred = kstep + 1 + lb;
    double O = 1e16, P = 1e16;
    const int end = pr.first + pr.nb;
    for (int c = pr.first + (int)(threadIdx.x & 63); c < end; c += 64) {
        const double o = term_old(a, c);
        O = smin(O, o);
        P = smin(P, c < block ? term_pre<R, PRE_CHECK>(a, nb_all, c) : o);
    }
    O = wave_min(O);
    P = wave_min(P);
    const double cf = cfl_eff(a.cfl, kpred);
    dt_step = cfl_eff(a.cfl, kstep) * O;
    dt_pred = cf * P;
    const double spec = cf * O;
    const bool g = a.fixed[block] != 0u;
    const double used = g ? cf * smin(1e16, mg) : spec;
    a.skip_next[block] = spec != dt_pred ? 1u : 0u;   // the same value from every wave
    return (!g && a.skip[block] != 0u) || used != dt_pred;
}

}  // namespace hf
