// Face fluxes of cent_keep<2>, pressure_diss_lr and visc_lr on values already
// at hand (the LDS windows of the face-once kernels), in the reference's
// expression order (navier-stokes/convective.h:117-184, 212-245; viscous.h:
// 39-112; omni/infos/info_gradient.h:45-81).  Shared by flux_fast.hip and the
// tiled kernel (flux_tile.hpp); compiled without contraction.
#pragma once
#include "spd_internal.hpp"
#include "pow_series.hpp"
#include <cmath>

namespace spd {
namespace {

struct FastCfg
{
    double R, gm1;                  // gas constant, gamma - 1
    double spec_heat;               // gamma R / (gamma - 1)
    double half_RR, inv_gamma;      // 0.5 (R + R), 1 / (0.5 (gamma + gamma))
    // viscous law, pre-multiplied by the composition scale s (8 with cent_keep<2>, else 1)
    double mu_s, visc2_s, cond_s;   // constant law: s mu, s beta, s cp alpha
    double mu_ref_s, T_ref, inv_T_ref, power, prandtl, inv_prandtl;
    int    t_ref_one;               // T_ref == 1: T/T_ref == T exactly
    PowSeries ps;                   // (T/T_ref)^power near T = T_ref
    // pressure diffusion, sensor pre-multiplied by s
    double scl_s, ducros_eps, ducros_s, eps_p, eps_T;
};

// The gas and the terms of a descriptor, with the composition scale sc (8 with
// cent_keep<2>, whose flux is formed times 8, else 1) multiplied in
inline void cfg_gas(FastCfg& C, const spd_flux_desc& f)
{
    C.R = f.R;
    C.gm1 = f.gamma - 1.0;
    C.spec_heat = f.gamma*f.R/(f.gamma - 1.0);
    C.half_RR = 0.5*(f.R + f.R);
    C.inv_gamma = 1.0/(0.5*(f.gamma + f.gamma));
}

inline void cfg_pdiss(FastCfg& C, const spd_flux_term& t, double sc)
{
    C.scl_s = sc*t.sensor_param; C.ducros_eps = t.sensor_param; C.ducros_s = sc;
    C.eps_p = t.eps_p; C.eps_T = t.eps_T;
}

// A constant divisor and its reciprocal for div_const, which takes no infinite
// one (its residual would be 0*inf): 1 with the reciprocal 0 gives the 0 of
// a/inf (an infinite Prandtl number switches heat conduction off)
inline void const_divisor(double b, double& d, double& y)
{
    const bool inf = std::isinf(b);
    d = inf ? 1.0 : b;
    y = inf ? 0.0 : 1.0/b;
}

inline void cfg_visc(FastCfg& C, const spd_flux_term& t, double sc)
{
    // constant law (viscous_laws.h:77-99): beta = -2 mu / 3, alpha = mu / Pr
    C.mu_s = sc*t.mu;
    C.visc2_s = sc*double(-2.0*t.mu/3.0);
    C.cond_s = C.spec_heat*(sc*(t.mu*(1.0/t.prandtl)));
    // power law (viscous_laws.h:121-134)
    C.mu_ref_s = sc*t.mu; C.power = t.power;
    const_divisor(t.T_ref, C.T_ref, C.inv_T_ref);
    const_divisor(t.prandtl, C.prandtl, C.inv_prandtl);
    C.t_ref_one = (t.T_ref == 1.0);
    C.ps = PowSeries::make(t.power);
}

struct CellV { double p, T, u, v, w, rho, e; };

template <int D> __device__ inline double vel(const CellV& c) { return D == 0 ? c.u : (D == 1 ? c.v : c.w); }

// a/b, rounded as the IEEE quotient, where b and the quotient are well inside
// the normal range (1e-290 to 1e290): the reciprocal instruction (relative
// error e <= 2^-22) times 1 + e + e^2 is good to e^3, and one residual step
// rounds the quotient.  7 instructions; the compiler's division adds two
// scalings and a choice for the ends of the range, and a fix-up of special
// values, which quot_inf keeps.  With these a 256^3 {KEEP2, power law} grid
// takes 480 us, 489 with the compiler's divisions, a fused step 2.11 ms, 2.15.
__device__ inline double quot(double a, double b)
{
    double y = __builtin_amdgcn_rcp(b);
    const double e = __builtin_fma(-b, y, 1.0);
    y = __builtin_fma(y, __builtin_fma(e, e, e), y);
    const double q = a*y;
    return __builtin_fma(__builtin_fma(-q, b, a), y, q);
}

// the same with the division's results for zeros, infinities and NaN
__device__ inline double quot_inf(double a, double b) { return __builtin_amdgcn_div_fixup(quot(a, b), b, a); }

__device__ inline CellV make_cell(const FastCfg& C, double p, double T, double u, double v, double w)
{
    CellV c{p, T, u, v, w, 0.0, 0.0};
    c.rho = quot_inf(p, C.R*T);
    c.e   = quot_inf(p, c.rho*C.gm1);
    return c;
}

// a / b, correctly rounded, for b a constant with y = RN(1/b) (Markstein's
// correction step: q0 = a y, r = a - b q0 exactly, q = q0 + r y)
__device__ inline double div_const(double a, double b, double y)
{
    const double q0 = a*y;
    const double r = __builtin_fma(-q0, b, a);
    return __builtin_fma(r, y, q0);
}

// the same with the division's results for an infinite a
__device__ inline double div_const_inf(double a, double b, double y)
{
    return __builtin_amdgcn_div_fixup(div_const(a, b, y), b, a);
}

// (T/T_ref)^n of the power law for N faces of a thread, from the sums of the
// temperatures at their sides: by the branch-free binomial series, and where a
// lane's x is outside its range by the library pow -- one cold loop behind a
// wave-uniform branch, placed where little else is live, so that the hot path
// keeps its registers and no later launch has to complete a block.  (A launch
// for that after every flux_div and stage cost 4-8 us and a gap even with
// nothing to do: 64^3 ten steps 754 -> 670 us without it, channel ten steps
// 5.81 -> 5.10 ms, channel flux_div 128.5 -> 117.5 us, with the shallower
// prefetch of the 16 x 16 kernel that makes room for it.)  Every kernel evaluates a face's x^n this way, so a face has
// the same bits whichever kernel evaluates it.
// Faces from M on are evaluated where `more` (the same in a whole wave) says so.
template <int M, int N>
__device__ inline void pow_faces(const PowSeries& ps, const double (&x)[N], double n, bool more, double (&pw)[N])
{
    bool bad = false;
    #pragma unroll
    for (int e = 0; e < M; ++e)
    {
        bad |= !ps.in_range(x[e]);
        pw[e] = ps.eval(x[e]);
    }
    if (M < N && more)
    {
        #pragma unroll
        for (int e = M; e < N; ++e)
        {
            bad |= !ps.in_range(x[e]);
            pw[e] = ps.eval(x[e]);
        }
    }
    if (__builtin_expect(__any(bad), 0))
    {
        #pragma clang loop unroll(disable)
        for (int f = 0; f < N; ++f)
        {
            double xf = x[0];
            #pragma unroll
            for (int e = 1; e < N; ++e) xf = f == e ? x[e] : xf;
            if (ps.in_range(xf)) continue;
            const double r = pow(xf, n);
            #pragma unroll
            for (int e = 0; e < N; ++e) pw[e] = f == e ? r : pw[e];
        }
    }
}

// x = T/T_ref of a face
__device__ inline double pow_arg(const FastCfg& C, double ST)
{
    const double Tf = ST*0.5;
    return C.t_ref_one ? Tf : div_const(Tf, C.T_ref, C.inv_T_ref);
}

// ducros_t::get_sensor (state_sensor.h:32-42); g[c][q], q = u, v, w
__device__ inline double ducros(const double g[3][3], double eps)
{
    double theta_sq = g[0][0] + g[1][1] + g[2][2];
    theta_sq *= theta_sq;
    const double v0 = g[1][2] - g[2][1];
    const double v1 = g[2][0] - g[0][2];
    const double v2 = g[0][1] - g[1][0];
    const double vort_sq = v0*v0 + v1*v1 + v2*v2;
    return theta_sq/(theta_sq + vort_sq + eps);
}

// Sums shared by the terms of one face: SU = uL+uR (= 2 u_face) etc.
struct FaceSums { double SU, SV, SW, SP, ST, K; };

__device__ inline FaceSums face_sums(const CellV& L, const CellV& R)
{
    FaceSums f;
    f.SU = L.u + R.u; f.SV = L.v + R.v; f.SW = L.w + R.w;
    f.SP = L.p + R.p; f.ST = L.T + R.T;
    f.K  = L.u*R.u + L.v*R.v + L.w*R.w;
    return f;
}

// pressure_diss_lr (convective.h:212-245), times the composition scale s:
// every output is a product chain that starts with the sensor value, so a
// sensor pre-multiplied by s (a power of two) scales every output exactly.
template <int SENSOR>
__device__ inline void pdiss_s(const FastCfg& C, const CellV& L, const CellV& R, const FaceSums& f,
                               const double g[3][3], double F[5])
{
    const double delta_p = L.p - R.p;
    const double delta_T = L.T - R.T;
    const double pavg = 0.5*f.SP;
    const double Tavg = 0.5*f.ST;
    const double inv_RT = 1.0/(C.half_RR*Tavg);
    const double p_inv_rt2 = pavg*inv_RT/Tavg;
    const double k = 0.5*f.K;
    const double u = 0.5*f.SU, v = 0.5*f.SV, w = 0.5*f.SW;
    const double scl = (SENSOR == SPD_SENSOR_DUCROS) ? C.ducros_s*ducros(g, C.ducros_eps) : C.scl_s;
    const double a = scl*C.eps_p*delta_p;
    const double b = scl*C.eps_T*delta_T*p_inv_rt2;
    F[0] = a*inv_RT - b;
    F[1] = a*(k*inv_RT + C.inv_gamma) - b*(0.5*k);
    F[2] = a*u*inv_RT - b*u;
    F[3] = a*v*inv_RT - b*v;
    F[4] = a*w*inv_RT - b*w;
}

template <int KEEP, int PDISS, int VISC> struct Spec
{
    static constexpr bool keep = KEEP != 0;
    static constexpr bool pd = PDISS != 0;           // 1 + sensor kind
    static constexpr int sensor = PDISS - 1;
    static constexpr bool vs = VISC != 0;             // 1 + law, + 2 with the WALE subgrid model
    static constexpr int law = (VISC - 1) & 1;
    static constexpr bool wale = VISC > 2;
    static constexpr bool full_grad = (pd && sensor == SPD_SENSOR_DUCROS) || wale;
};

// WALE subgrid viscosity of a face (subgrid_scale.h:44-84) from its full
// velocity gradient g[c][q] = d u_q / d x_c and face p, T; the sums in the
// order of wale_mu_t in flux_cell.hpp
template <class Cfg>
__device__ inline double wale_s(const Cfg& C, double pf, double Tf, const double g[3][3])
{
    const double rho = pf/(C.R*Tf);
    double g2[3][3], sd[3][3], s[3][3];
    #pragma unroll
    for (int j = 0; j < 3; ++j)
        #pragma unroll
        for (int i = 0; i < 3; ++i) g2[i][j] = g[0][i]*g[j][0] + g[1][i]*g[j][1] + g[2][i]*g[j][2];
    #pragma unroll
    for (int j = 0; j < 3; ++j)
        #pragma unroll
        for (int i = 0; i < 3; ++i)
        {
            sd[i][j] = 0.5*(g2[i][j] + g2[j][i]);
            s[i][j]  = 0.5*(g[j][i] + g[i][j]);
        }
    double tr = 0.0;
    #pragma unroll
    for (int d = 0; d < 3; ++d) tr += 0.33333333333333333*g2[d][d];
    #pragma unroll
    for (int d = 0; d < 3; ++d) sd[d][d] -= tr;
    double ssd = 0.0, ss = 0.0;
    #pragma unroll
    for (int j = 0; j < 3; ++j)
        #pragma unroll
        for (int i = 0; i < 3; ++i) ssd += sd[i][j]*sd[i][j];
    #pragma unroll
    for (int j = 0; j < 3; ++j)
        #pragma unroll
        for (int i = 0; i < 3; ++i) ss += s[i][j]*s[i][j];
    const double r0 = sqrt(ssd), r1 = sqrt(r0), r2 = sqrt(ss);
    return rho*C.sgs_cw*C.sgs_cw*C.sgs_delta*C.sgs_delta*ssd*r0/(1e-8 + ss*ss*r2 + ssd*r1);
}

// visc_lr row D for the unit normal of identity coordinates (viscous.h:39-112),
// times the composition scale s (carried by mu, beta and the conductivity);
// pw: the face's (T/T_ref)^n (pow_faces) with the power law.
template <int D, class S, bool MAP, class Cfg>
__device__ inline void visc_s(const Cfg& C, const FaceSums& f, const double g[3][3], double gT, double nf,
                              double F[5], double pw)
{
    double mu, visc2, cond;
    if constexpr (S::law == SPD_LAW_POWER)
    {
        mu    = C.mu_ref_s*pw;
        visc2 = -0.66666666667*mu;
        cond  = C.spec_heat*div_const(mu, C.prandtl, C.inv_prandtl);
    }
    else
    {
        mu = C.mu_s; visc2 = C.visc2_s; cond = C.cond_s;
    }
    if constexpr (S::wale)
    {
        // sgs_visc_t (viscous_laws.h:186-196): mu + mu_t, beta - 0.666.. mu_t,
        // alpha + mu_t / Pr_t, all times the composition scale
        const double mu_t = C.scale*wale_s(C, 0.5*f.SP, 0.5*f.ST, g);
        const double alpha = (S::law == SPD_LAW_POWER ? div_const(mu, C.prandtl, C.inv_prandtl) : C.alpha_s)
                             + mu_t/C.sgs_prt;
        cond  = C.spec_heat*alpha;
        visc2 = visc2 - 0.66666666667*mu_t;
        mu    = mu + mu_t;
    }
    const double div = g[0][0] + g[1][1] + g[2][2];
    double t[3];
    #pragma unroll
    for (int b = 0; b < 3; ++b)
    {
        if (b == D) t[b] = mu*(g[D][D] + g[D][D]) + visc2*div;
        else if (D < b) t[b] = mu*(g[D][b] + g[b][D]);
        else            t[b] = mu*(g[b][D] + g[D][b]);
    }
    // (uf t0 + vf t1 + wf t2) with uf = SU/2: the halving is exact
    const double hsum = 0.5*(f.SU*t[0] + f.SV*t[1] + f.SW*t[2]);
    const double ht = hsum + cond*gT;
    F[0] = 0.0;
    if constexpr (MAP)
    {
        // -(n . ht), -(n . tau) with the area-weighted face normal n = nf e_D
        F[1] = -(nf*ht);
        F[2] = -(nf*t[0]);
        F[3] = -(nf*t[1]);
        F[4] = -(nf*t[2]);
    }
    else
    {
        F[1] = -ht;
        F[2] = -t[0];
        F[3] = -t[1];
        F[4] = -t[2];
    }
}

// Face product P = F / dx with F = keep + (pdiss + visc) composed in the
// reference's order (omni/compose.h:19-24) and flux_div_basic's scaling
// (flux_div_basic.h:66-68).  cent_keep<2> (convective.h:117-184) is written
// with its power-of-two factors pulled out: with CX = (rhoL+rhoR)(unR+unL),
// continuity = CX/4 and the other outputs are 1/8 of
//   energy:   CX K + CX (eL+eR) + 4 (unL pR + unR pL)
//   momentum: CX (qL+qR) + 4 (pL+pR) n
// Every factor is a power of two, so each rounding equals the reference's;
// the other terms are evaluated pre-multiplied by 8 and the factor is folded
// into 1/dx.
// On mapped (diagonal) coordinates (MAP) the normals enter: mt = {n_D of the
// left cell, n_D of the right cell, n_D of the face} (metric(), the area
// factors of coord_system.h:250-267), u_n = u_D n_D (the other components of a
// diagonal normal are zero); the result is then the flux scaled by the
// composition scale, not yet by 1/dx: the cells apply their own
// jac (1 - 2 pm)/dx (flux_div_basic.h:66-68).
template <int D, class S, bool MAP, class Cfg>
__device__ inline void face_product(const Cfg& C, const CellV& L, const CellV& R, const double g[3][3], double gT,
                                    double idx, const double mt[3], double P[5], double pw)
{
    const FaceSums f = face_sums(L, R);
    double s8[5];
    if (S::vs) visc_s<D, S, MAP>(C, f, g, gT, mt[2], s8, pw);
    if (S::pd)
    {
        double z[5];
        pdiss_s<S::sensor>(C, L, R, f, g, z);
        if (S::vs) { for (int n = 0; n < 5; ++n) s8[n] = z[n] + s8[n]; }
        else       { for (int n = 0; n < 5; ++n) s8[n] = z[n]; }
    }
    if (S::keep)
    {
        double unL = vel<D>(L), unR = vel<D>(R);
        if constexpr (MAP) { unL = unL*mt[0]; unR = unR*mt[1]; }
        const double CX = (L.rho + R.rho)*(unR + unL);
        const double Ep = CX*f.K + CX*(L.e + R.e) + 4.0*(unL*R.p + unR*L.p);
        double M[3] = {CX*f.SU, CX*f.SV, CX*f.SW};
        if constexpr (MAP) M[D] = M[D] + 4.0*(f.SP*mt[2]);
        else               M[D] = M[D] + 4.0*f.SP;
        if constexpr (MAP)
        {
            // 8 F: continuity 2 CX (+ s8), the others as below; the cells scale by 1/8
            if (S::vs || S::pd)
            {
                P[0] = S::pd ? 2.0*(CX + 0.5*s8[0]) : 2.0*CX;
                P[1] = Ep + s8[1]; P[2] = M[0] + s8[2]; P[3] = M[1] + s8[3]; P[4] = M[2] + s8[4];
            }
            else
            {
                P[0] = 2.0*CX; P[1] = Ep; P[2] = M[0]; P[3] = M[1]; P[4] = M[2];
            }
            return;
        }
        const double i4 = 0.25*idx, i8 = 0.125*idx;
        if (S::vs || S::pd)
        {
            P[0] = S::pd ? (CX + 0.5*s8[0])*i4 : CX*i4;
            P[1] = (Ep + s8[1])*i8;
            P[2] = (M[0] + s8[2])*i8;
            P[3] = (M[1] + s8[3])*i8;
            P[4] = (M[2] + s8[4])*i8;
        }
        else
        {
            P[0] = CX*i4; P[1] = Ep*i8; P[2] = M[0]*i8; P[3] = M[1]*i8; P[4] = M[2]*i8;
        }
    }
    else
    {
        #pragma unroll
        for (int n = 0; n < 5; ++n) P[n] = MAP ? s8[n] : s8[n]*idx;
    }
}

// info::gradient on mapped coordinates (omni/infos/info_gradient.h, the
// coordinate scaling of face_grad): component a of every gradient divided by
// d x_a / d xi_a at the face point (mn for the face normal axis D, the cell
// centre values mt1 / mt2 for the other two); identity axes divide by 1.
template <int D>
__device__ inline void grads_map(const DevGeom& G, double g[3][3], double& gT, double mD, double mA, double mB)
{
    constexpr int A = (D + 1) % 3, B = (D + 2) % 3;
    if (G.map_kind[D] != SPD_MAP_IDENTITY) { for (int b = 0; b < 3; ++b) g[D][b] = g[D][b]/mD; gT = gT/mD; }
    if (G.map_kind[A] != SPD_MAP_IDENTITY) for (int b = 0; b < 3; ++b) g[A][b] = g[A][b]/mA;
    if (G.map_kind[B] != SPD_MAP_IDENTITY) for (int b = 0; b < 3; ++b) g[B][b] = g[B][b]/mB;
}

// The same when only y is mapped: m = d y / d eta at the face point and
// rm = RN(1/m), tabulated per block, so that each quotient costs four
// operations instead of a division (div_const: the same bits; the last one keeps
// an infinite gradient infinite, which div_const alone turns into NaN: 1 % of
// the 192 x 128 x 96 channel's flux_div, 107.6 -> 108.8 us)
template <int D>
__device__ inline void grads_map_y(double g[3][3], double& gT, double m, double rm)
{
    #pragma unroll
    for (int b = 0; b < 3; ++b) g[1][b] = div_const_inf(g[1][b], m, rm);
    if (D == 1) gT = div_const_inf(gT, m, rm);
}

// metric() of a diagonal map at a point with derivatives m0, m1, m2: jac =
// 1/(m0 m1 m2), normal component D = 1/(m_D jac) (core/coord_system.h:250-302)
__device__ inline double jac_at(double m0, double m1, double m2) { return 1.0/(m0*m1*m2); }
__device__ inline double nrm_at(double mD, double jac) { return 1.0/(mD*jac); }

// 0.25-weighted four-point tangential gradient (info_gradient.h:63-79):
// the reference sums r(0.25 q it) terms; 0.25 factors out exactly.
__device__ inline double tang(double a, double b, double c, double d, double it)
{
    return 0.25*(((a*it - b*it) + c*it) - d*it);
}

// normal gradient (info_gradient.h:63, 73): -qL/dx + qR/dx
__device__ inline double normal_grad(double qL, double qR, double id)
{
    return qR*id - qL*id;
}

} // namespace
} // namespace spd
