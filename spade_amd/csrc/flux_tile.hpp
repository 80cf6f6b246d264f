// Tiled flux_div for every composition with compile-time code, on blocks of
// any size and on identity or diagonal (mapped) coordinates.  It runs whatever
// the 16 x 16 kernel of flux_fast.hip does not take: cent_keep<4>, totani_lr,
// weno_t, fweno_t, first_order_t, weno_fds_t (each alone or followed by
// visc_lr), WALE viscosities, and cent_keep<2> / pressure_diss_lr / visc_lr on
// other block cross-sections.
//
// A workgroup owns a tile of wi x wj columns of a block (all of a small block)
// and a share of its planes, one thread per column, and marches over k.  Each
// face flux is evaluated once: a thread evaluates the low x-face, the low
// y-face and the high z-face of its cell, lanes of the last two waves add the
// tile's closing x- and y-faces, and a cell reads its high x- and y-faces from
// LDS.  The per-cell kernel this replaces evaluated six faces per cell, each
// gathering its stencil (and, mapped, its tanh metrics) again from memory
// through a run-time index, at one wave per SIMD.  Measured per flux_div,
// before and now: cent_keep<2> + visc_lr on 5 x 6 x 8 blocks of 24 x 20 x 12,
// 2549 -> 67 us; WENO + visc_lr on 128^3, 2594 -> 211 us; cent_keep<4> + WALE on
// 96^3 in 32^3 blocks, 602 -> 88 us; WENO + visc_lr on 80 x 48 x 64 stretched
// cells, 798 -> 43 us; twelve blocks of 4 x 8 x 4, 72.7 -> 6.8 us.
//
// LDS holds the velocities of planes k-1, k, k+1 (ring of three) and, of plane
// k, p, T and the per-cell quantities the composition's faces share (rho, e;
// the split coefficients of WENO): what a face needs of a neighbour is computed
// once per cell.  Records are interleaved per cell with an odd stride (3, and
// 3, 5 or 7 doubles), so a row of lanes reads LDS without bank conflicts and
// the offsets of a cell's x-neighbours and components are immediates.  With a
// 16 x 16 tile the window of the widest composition takes 73 KB, two workgroups per
// CU; longer and narrower tiles up to 90 KB, one.
//
// Arithmetic: the expressions of flux_cell.hpp in the same order, with the
// components of a diagonal map's face normal that are zero left out, so for
// finite states the result equals the per-cell code's bit for bit.  (The per-cell
// code multiplies those components by the velocities and the pressure, so around an
// infinite one it gives NaN at faces where this gives an infinity or, in the
// outputs that do not contain it, a number.)
#pragma once
#include "spd_internal.hpp"
#include "flux_face.hpp"
#include "flux_cell.hpp"
#include <algorithm>

namespace spd {
namespace {

struct TileCfg : FastCfg
{
    double scale, alpha_s;                 // composition scale; constant law's alpha times it
    double sgs_cw, sgs_delta, sgs_prt;     // WALE
    double gamma, gamma_R;
    int    split_phys, smooth;             // WENO
    // tiling: nominal tile columns and rows, tiles per block, workgroups along k
    int    wi, wj, tx, ty, zs;
};

// what the faces of a composition need of a cell, beyond p, T, u, v, w
template <int CONV, int PDISS, int VISC>
struct TileSpec : Spec<(CONV == CV_KEEP2), PDISS, VISC>
{
    using Base = Spec<(CONV == CV_KEEP2), PDISS, VISC>;
    static constexpr int conv = CONV;
    static constexpr bool wide = CONV == CV_KEEP4 || CONV == CV_WENO || CONV == CV_FWENO || CONV == CV_FDS;
    static constexpr int H = wide ? 2 : 1;                       // halo layers along the axes
    static constexpr bool grad = Base::vs || Base::full_grad;    // faces need velocity gradients
    static constexpr int extra = (CONV == CV_KEEP2 || CONV == CV_KEEP4 || CONV == CV_TOTANI) ? 2
                               : (CONV == CV_WENO || CONV == CV_FWENO || CONV == CV_FIRST) ? 4 : 0;
    static constexpr int SS = (2 + extra) | 1;                   // doubles per scalar record
    static constexpr bool power = Base::vs && Base::law == SPD_LAW_POWER;
    static constexpr double scale = CONV == CV_KEEP2 ? 8.0 : 1.0;
};

// x: KEEP / Totani {rho, e}; WENO, first order {rho/2, E, E + p/rho, sigma rho}
// (physical splitting: {rho/2, -, enthalpy, -}); FWENO {rho, E, E + p/rho, s}
struct TCell { double p, T, u, v, w, x[4]; };

template <int D> __device__ inline double vel(const TCell& c) { return D == 0 ? c.u : (D == 1 ? c.v : c.w); }

struct Raw5 { double p, T, u, v, w; };

template <class S>
__device__ inline TCell derive(const TileCfg& C, const Raw5& r)
{
    TCell c{r.p, r.T, r.u, r.v, r.w, {0.0, 0.0, 0.0, 0.0}};
    if constexpr (S::extra == 2)
    {
        c.x[0] = quot_inf(r.p, C.R*r.T);
        c.x[1] = quot_inf(r.p, c.x[0]*C.gm1);
    }
    else if constexpr (S::conv == CV_WENO || S::conv == CV_FIRST)
    {
        // rusanov_t / phys_flux_t (flux_funcs.h:19-52, 107-124)
        const double k2 = r.u*r.u + r.v*r.v + r.w*r.w;
        const double rho = quot_inf(r.p, C.R*r.T);
        const double pdiff = quot_inf(r.p, rho), ei = quot_inf(r.p, rho*C.gm1);
        c.x[0] = 0.5*rho;
        if (S::conv == CV_WENO && C.split_phys) c.x[2] = 0.5*k2 + pdiff + ei;
        else
        {
            c.x[1] = 0.5*k2 + ei;
            c.x[2] = c.x[1] + pdiff;
            c.x[3] = 0.5*(sqrt(k2) + sqrt(C.gamma_R*r.T))*rho;
        }
    }
    else if constexpr (S::conv == CV_FWENO)
    {
        // fweno_t (convective.h:355-496)
        const double k2 = r.u*r.u + r.v*r.v + r.w*r.w;
        const double RT = C.R*r.T;
        c.x[0] = quot_inf(r.p, RT);
        c.x[3] = (sqrt(k2) + sqrt(RT*C.gamma))*c.x[0]*0.5;
        c.x[1] = k2*0.5 + quot_inf(RT, C.gm1);
        c.x[2] = c.x[1] + RT;
    }
    return c;
}

// Output n of a cell's half flux through a face of direction D with area
// factor nc, and of its dissipation: the upwind / downwind split fluxes are
// their sum and difference (split_rusanov / split_phys of flux_cell.hpp; the
// physical splitting's x[3] is 0, and both parts are then the same flux)
template <int D>
__device__ inline double split_out(const TCell& q, double nc, double un, int n)
{
    if (n == 0) return q.x[0]*un;
    if (n == 1) return q.x[0]*un*q.x[2];
    const double f = q.x[0]*(n == 2 ? q.u : (n == 3 ? q.v : q.w))*un;
    return n == 2 + D ? f + 0.5*q.p*nc : f;
}

__device__ inline double split_diss(const TCell& q, int n)
{
    return n == 0 ? q.x[3] : q.x[3]*(n == 1 ? q.x[1] : (n == 2 ? q.u : (n == 3 ? q.v : q.w)));
}

// The candidate values of weno_t and fweno_t.  A product with 1/2 is exact, so
// fusing it into its sum leaves the one rounding of the per-cell expressions.
struct WenoR { double r0, r1, r2, r3; };
__device__ inline WenoR weno_candidates(double u0, double u1, double u2, double d1, double d2, double d3)
{
    return {__builtin_fma(-0.5, u0, 1.5*u1), __builtin_fma(0.5, u1, 0.5*u2),
            __builtin_fma(0.5, d1, 0.5*d2), __builtin_fma(-0.5, d3, 1.5*d2)};
}

__device__ inline double weno_lin(double u0, double u1, double u2, double d1, double d2, double d3)
{
    const WenoR r = weno_candidates(u0, u1, u2, d1, d2, d3);
    return (1.0/3.0)*r.r0 + (2.0/3.0)*r.r1 + (2.0/3.0)*r.r2 + (1.0/3.0)*r.r3;
}

// weno_t's smooth weights (convective.h:275-332).  The b are at least 1e-16,
// so the squares start at 1e-32 and the a end at 1e32: a division by a square
// needs the infinite case only, the weights' own divisions neither end.  That
// holds for squares up to 1e290 (split fluxes 1e72 apart) and for infinite ones
// (both a 0 is NaN either way); in the decade before overflow, where an a is
// subnormal, a weight may differ from the division's.  Six divisions
// a component were 40 % of the kernel's instructions: a 128^3 grid of
// {WENO, viscous} 247 -> 218 us with these, same bits.
__device__ inline double weno_smooth(double u0, double u1, double u2, double d1, double d2, double d3)
{
    const WenoR r = weno_candidates(u0, u1, u2, d1, d2, d3);
    const double eps = 1e-16;
    const double b0 = (u0 - u1)*(u0 - u1) + eps, b1 = (u1 - u2)*(u1 - u2) + eps;
    const double b2 = (d1 - d2)*(d1 - d2) + eps, b3 = (d2 - d3)*(d2 - d3) + eps;
    const double a0 = quot_inf(1.0/3.0, b0*b0), a1 = quot_inf(2.0/3.0, b1*b1);
    const double a2 = quot_inf(2.0/3.0, b2*b2), a3 = quot_inf(1.0/3.0, b3*b3);
    const double w0 = quot(a0, a0 + a1), w1 = 1.0 - w0, w2 = quot(a2, a2 + a3), w3 = 1.0 - w2;
    return w0*r.r0 + w1*r.r1 + w2*r.r2 + w3*r.r3;
}

// fweno_t's smooth weights (the same ratios with fewer divisions; a square
// that overflows gives its side the weight 0 or NaN, as the division does)
__device__ inline double fweno_smooth(double u0, double u1, double u2, double d1, double d2, double d3)
{
    const WenoR r = weno_candidates(u0, u1, u2, d1, d2, d3);
    const double eps = 1e-16;
    double a[4] = {u0 - u1, u1 - u2, d1 - d2, d2 - d3};
    #pragma unroll
    for (int n = 0; n < 4; ++n) { a[n] *= a[n]; a[n] += eps; a[n] *= a[n]; }
    const double w0 = quot_inf(a[1], a[0] + a[0] + a[1]), w3 = quot_inf(a[2], a[3] + a[3] + a[2]);
    return w0*r.r0 + (1.0 - w0)*r.r1 + (1.0 - w3)*r.r2 + w3*r.r3;
}

// cfd_coeff(i, 4) of flux_cell.hpp
constexpr double kKeep4A = (2.0/6.0)*(2.0/1.0)*1/1.0, kKeep4B = (2.0/24.0)*(2.0/1.0)*-1/2.0;

// Composed flux F (times S::scale) through a face of direction D.  q[0..n-1]:
// the cells at offsets -1, 0 (narrow) or -2 .. 1 (wide); nc: their normal
// factors, nf: the face's (all 1 on identity coordinates); g, gT: the face
// gradient and pw the power law's (T/T_ref)^n where the composition has them.
template <int D, class S>
__device__ inline void visc_face(const TileCfg& C, const TCell& A, const TCell& B, double nf, const double g[3][3],
                                 double gT, double z[5], double pw)
{
    FaceSums f;
    f.SU = A.u + B.u; f.SV = A.v + B.v; f.SW = A.w + B.w;
    f.SP = A.p + B.p; f.ST = A.T + B.T; f.K = 0.0;
    visc_s<D, S, true>(C, f, g, gT, nf, z, pw);
}

template <int D, class S>
__device__ inline void face_flux(const TileCfg& C, const TCell* q, const double* nc, double nf, const double g[3][3],
                                 double gT, double F[5], double pw)
{
    constexpr int l = S::wide ? 1 : 0, r = l + 1;
    const TCell& A = q[l];
    const TCell& B = q[r];
    // the viscous part first: its gradients are then dead before the wide
    // stencils' arithmetic
    double z[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if constexpr (S::vs && S::conv != CV_KEEP2 && S::conv != CV_NONE)
    {
        visc_face<D, S>(C, A, B, nf, g, gT, z, pw);
        if constexpr (S::wide)
        {
            #pragma unroll
            for (int n = 1; n < 5; ++n) keep_here(z[n]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if constexpr (S::conv == CV_KEEP2 || S::conv == CV_NONE)
    {
        const CellV L{A.p, A.T, A.u, A.v, A.w, A.x[0], A.x[1]}, R{B.p, B.T, B.u, B.v, B.w, B.x[0], B.x[1]};
        const double mt[3] = {nc[l], nc[r], nf};
        face_product<D, S, true>(C, L, R, g, gT, 1.0, mt, F, pw);
        return;
    }
    else if constexpr (S::conv == CV_TOTANI)
    {
        const double unl = vel<D>(A)*nc[l], unr = vel<D>(B)*nc[r];
        const double c = 0.25*(A.x[0] + B.x[0])*(unl + unr);
        F[0] = c;
        F[1] = 0.5*c*(A.x[1] + B.x[1] + A.u*B.u + A.v*B.v + A.w*B.w) + 0.5*(unl*B.p + unr*A.p);
        F[2] = 0.5*c*(A.u + B.u);
        F[3] = 0.5*c*(A.v + B.v);
        F[4] = 0.5*c*(A.w + B.w);
        F[2 + D] = F[2 + D] + 0.5*(nc[l]*A.p + nc[r]*B.p);
    }
    else if constexpr (S::conv == CV_KEEP4)
    {
        double un[4];
        #pragma unroll
        for (int m = 0; m < 4; ++m) un[m] = vel<D>(q[m])*nc[m];
        double c = 0.0, mx = 0.0, my = 0.0, mz = 0.0, gp = 0.0, k = 0.0, ie = 0.0, pp = 0.0;
        #pragma unroll
        for (int ii = 1; ii <= 2; ++ii)
        {
            const double a = ii == 1 ? kKeep4A : kKeep4B;
            #pragma unroll
            for (int jj = 0; jj < ii; ++jj)
            {
                const int i0 = 1 - jj, i1 = i0 + ii;
                const TCell& X = q[i0];
                const TCell& Y = q[i1];
                const double cl = a*(0.25*(X.x[0] + Y.x[0])*(un[i1] + un[i0]));
                c  += cl;
                mx += cl*(0.5*(X.u + Y.u));
                my += cl*(0.5*(X.v + Y.v));
                mz += cl*(0.5*(X.w + Y.w));
                gp += a*(0.5*(X.p + Y.p));
                k  += 0.5*cl*(X.u*Y.u + X.v*Y.v + X.w*Y.w);
                ie += cl*(0.5*(X.x[1] + Y.x[1]));
                pp += a*(0.5*(un[i0]*Y.p + un[i1]*X.p));
            }
        }
        double m[3] = {mx, my, mz};
        m[D] = m[D] + gp*nf;
        F[0] = 2.0*c;
        F[1] = 2.0*(k + ie + pp);
        F[2] = 2.0*m[0]; F[3] = 2.0*m[1]; F[4] = 2.0*m[2];
    }
    else if constexpr (S::conv == CV_FIRST)
    {
        const double ul = vel<D>(A)*nc[l], ur = vel<D>(B)*nc[r];
        #pragma unroll
        for (int n = 0; n < 5; ++n)
            F[n] = (split_out<D>(A, nc[l], ul, n) + split_diss(A, n)) + (split_out<D>(B, nc[r], ur, n) - split_diss(B, n));
    }
    else if constexpr (S::conv == CV_WENO)
    {
        // one output at a time: its six split fluxes and weights are dead
        // before the next one's
        double un[4];
        #pragma unroll
        for (int m = 0; m < 4; ++m) un[m] = vel<D>(q[m])*nc[m];
        #pragma unroll
        for (int n = 0; n < 5; ++n)
        {
            double up[3], dn[3];
            #pragma unroll
            for (int m = 0; m < 4; ++m)
            {
                const double sp = split_out<D>(q[m], nc[m], un[m], n), sg = split_diss(q[m], n);
                if (m < 3) up[m] = sp + sg;
                if (m > 0) dn[m - 1] = sp - sg;
            }
            F[n] = C.smooth ? weno_smooth(up[0], up[1], up[2], dn[0], dn[1], dn[2])
                            : weno_lin(up[0], up[1], up[2], dn[0], dn[1], dn[2]);
            keep_here(F[n]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    else if constexpr (S::conv == CV_FWENO)
    {
        double fl[4], ds[4], un[4];
        auto apply = [&](int n)
        {
            const double u0 = fl[0] + ds[0], u1 = fl[1] + ds[1], u2 = fl[2] + ds[2];
            const double d1 = fl[1] - ds[1], d2 = fl[2] - ds[2], d3 = fl[3] - ds[3];
            F[n] = C.smooth ? fweno_smooth(u0, u1, u2, d1, d2, d3) : weno_lin(u0, u1, u2, d1, d2, d3);
        };
        #pragma unroll
        for (int m = 0; m < 4; ++m) { un[m] = vel<D>(q[m])*nc[m]; fl[m] = un[m]*(0.5*q[m].x[0]); ds[m] = q[m].x[3]; }
        apply(0);
        #pragma unroll
        for (int m = 0; m < 4; ++m) { fl[m] *= q[m].x[2]; ds[m] *= q[m].x[1]; }
        apply(1);
        #pragma unroll
        for (int dr = 0; dr < 3; ++dr)
        {
            #pragma unroll
            for (int m = 0; m < 4; ++m)
            {
                const double vd = dr == 0 ? q[m].u : (dr == 1 ? q[m].v : q[m].w);
                fl[m] = un[m]*q[m].x[0]*vd;
                if (dr == D) fl[m] = fl[m] + q[m].p*nc[m];
                fl[m] *= 0.5;
                ds[m] = q[m].x[3]*vd;
            }
            apply(2 + dr);
        }
    }
    else if constexpr (S::conv == CV_FDS)
    {
        // weno_fds_t<rusanov_fds_t> (f_weno_fds in flux_cell.hpp)
        double qa[4][5];
        #pragma unroll
        for (int m = 0; m < 4; ++m)
        {
            qa[m][0] = q[m].p; qa[m][1] = q[m].T; qa[m][2] = q[m].u; qa[m][3] = q[m].v; qa[m][4] = q[m].w;
        }
        double ql[5], qr[5], qf[5];
        #pragma unroll
        for (int n = 0; n < 5; ++n)
        {
            ql[n] = 0.5*qa[1][n] + 0.5*qa[2][n];
            qr[n] = ql[n];
            if (!C.smooth)
            {
                ql[n] *= 2.0/3.0;
                qr[n] *= 2.0/3.0;
                ql[n] += (1.0/3.0)*(-0.5*qa[0][n] + 1.5*qa[1][n]);
                qr[n] += (1.0/3.0)*(1.5*qa[2][n] - 0.5*qa[3][n]);
            }
            qf[n] = (qa[1][n] + qa[2][n])*0.5;
        }
        const double un = nf*qf[2 + D];
        const double rl = ql[0]/(C.R*ql[1]), rr = qr[0]/(C.R*qr[1]);
        const double el = 0.5*(ql[2]*ql[2] + ql[3]*ql[3] + ql[4]*ql[4]) + ql[0]/(rl*C.gm1);
        const double er = 0.5*(qr[2]*qr[2] + qr[3]*qr[3] + qr[4]*qr[4]) + qr[0]/(rr*C.gm1);
        const double sg = un + sqrt(C.gamma_R*qf[1]);
        const double sl = sg*rl, sr = sg*rr;
        F[0] = sl - sr;
        F[1] = sl*el - sr*er;
        #pragma unroll
        for (int n = 2; n < 5; ++n) F[n] = sl*ql[n] - sr*qr[n];
    }
    if constexpr (S::vs)
    {
        #pragma unroll
        for (int n = 1; n < 5; ++n) F[n] = F[n] + z[n];
    }
}

// Velocity planes k-1, k, k+1 of the window (3 doubles per cell; py: a row)
struct Win { const double *m, *z, *p; int py; };

// Face gradients from the window (info_gradient.h:45-81); a: element of the
// left cell, b: of the right one
template <class S>
__device__ inline void tile_grads_x(const Win& W, int a, const TCell& L, const TCell& R, double ix, double iy,
                                    double iz, double g[3][3], double& gT)
{
    const int b = a + 3, py = W.py;
    g[0][0] = normal_grad(L.u, R.u, ix); g[0][1] = normal_grad(L.v, R.v, ix); g[0][2] = normal_grad(L.w, R.w, ix);
    gT      = normal_grad(L.T, R.T, ix);
    g[1][0] = tang(W.z[a + py], W.z[a - py], W.z[b + py], W.z[b - py], iy);
    g[1][1] = tang(W.z[a + py + 1], W.z[a - py + 1], W.z[b + py + 1], W.z[b - py + 1], iy);
    g[1][2] = S::full_grad ? tang(W.z[a + py + 2], W.z[a - py + 2], W.z[b + py + 2], W.z[b - py + 2], iy) : 0.0;
    g[2][0] = tang(W.p[a], W.m[a], W.p[b], W.m[b], iz);
    g[2][1] = S::full_grad ? tang(W.p[a + 1], W.m[a + 1], W.p[b + 1], W.m[b + 1], iz) : 0.0;
    g[2][2] = tang(W.p[a + 2], W.m[a + 2], W.p[b + 2], W.m[b + 2], iz);
}

template <class S>
__device__ inline void tile_grads_y(const Win& W, int a, const TCell& L, const TCell& R, double ix, double iy,
                                    double iz, double g[3][3], double& gT)
{
    const int b = a + W.py;
    g[1][0] = normal_grad(L.u, R.u, iy); g[1][1] = normal_grad(L.v, R.v, iy); g[1][2] = normal_grad(L.w, R.w, iy);
    gT      = normal_grad(L.T, R.T, iy);
    g[2][0] = S::full_grad ? tang(W.p[a], W.m[a], W.p[b], W.m[b], iz) : 0.0;
    g[2][1] = tang(W.p[a + 1], W.m[a + 1], W.p[b + 1], W.m[b + 1], iz);
    g[2][2] = tang(W.p[a + 2], W.m[a + 2], W.p[b + 2], W.m[b + 2], iz);
    g[0][0] = tang(W.z[a + 3], W.z[a - 3], W.z[b + 3], W.z[b - 3], ix);
    g[0][1] = tang(W.z[a + 4], W.z[a - 2], W.z[b + 4], W.z[b - 2], ix);
    g[0][2] = S::full_grad ? tang(W.z[a + 5], W.z[a - 1], W.z[b + 5], W.z[b - 1], ix) : 0.0;
}

// sL, sR: the planes below and above the face
template <class S>
__device__ inline void tile_grads_z(const double* sL, const double* sR, int py, int a, const TCell& L, const TCell& R,
                                    double ix, double iy, double iz, double g[3][3], double& gT)
{
    g[2][0] = normal_grad(L.u, R.u, iz); g[2][1] = normal_grad(L.v, R.v, iz); g[2][2] = normal_grad(L.w, R.w, iz);
    gT      = normal_grad(L.T, R.T, iz);
    g[0][0] = tang(sL[a + 3], sL[a - 3], sR[a + 3], sR[a - 3], ix);
    g[0][1] = S::full_grad ? tang(sL[a + 4], sL[a - 2], sR[a + 4], sR[a - 2], ix) : 0.0;
    g[0][2] = tang(sL[a + 5], sL[a - 1], sR[a + 5], sR[a - 1], ix);
    g[1][0] = S::full_grad ? tang(sL[a + py], sL[a - py], sR[a + py], sR[a - py], iy) : 0.0;
    g[1][1] = tang(sL[a + py + 1], sL[a - py + 1], sR[a + py + 1], sR[a - py + 1], iy);
    g[1][2] = tang(sL[a + py + 2], sL[a - py + 2], sR[a + py + 2], sR[a - py + 2], iy);
}

// LDS of a tile launch in doubles, in the order the kernel lays it out
struct TileLds
{
    int hp, plane, sca, fx, fy, tab, total;
    __host__ __device__ TileLds(int wi, int wj, int share, int H, int SS, bool map)
    {
        hp = (wi + 2*H)*(wj + 2*H);
        plane = 3*hp;
        sca = 3*plane;                        // after three velocity planes
        fx = sca + SS*hp;
        fy = fx + 5*(wi + 1)*wj;
        tab = fy + 5*wi*(wj + 1);
        total = tab;
        if (map) total += (wi + 2*H) + 5*(wj + 2*H) + (share + 2*H + 1) + (wi + 1) + 3*(wj + 1) + (share + 1);
    }
};

// MAP: 0 identity coordinates, 1 only y mapped, 2 any diagonal map
template <class S, int MAP>
__global__ void __launch_bounds__(256, 2) __attribute__((flatten))
k_flux_div_spec_tile(DevGeom G, const double* __restrict__ prims, double* __restrict__ rhs, TileCfg C, int increment)
{
    extern __shared__ double lds[];
    constexpr int H = S::H, SS = S::SS, NQ = S::wide ? 4 : 2, l = S::wide ? 1 : 0;
    constexpr double sc = 1.0/S::scale;
    constexpr int Y = 2*H + 1;                // (z tables start at plane k0 - H)
    const int tid = threadIdx.x;
    // thread number of the halo columns and the closing faces.  Wide stencils
    // and WALE, whose waves with a fourth face bind the SIMD they run on, take
    // closing faces in waves 1 and 3 and halo columns in 0 and 2: the two
    // workgroups of a CU are placed one SIMD on from each other, so each SIMD
    // then holds one such wave, where of waves 2 and 3 one SIMD held two
    // ({WENO, viscous} 128^3 217 -> 212 us, {KEEP4, WALE} 96^3 91.2 -> 88.3).
    // The lighter KEEP2 kernels wait for memory instead and keep waves 2 and
    // 3 (67.4 us against 68.2 on 24x20x12 blocks).
    constexpr bool heavy = S::wide || S::wale;
    const int rt = heavy && blockDim.x == 256 ? (tid & 63) | ((tid & 64) << 1) | ((tid & 128) >> 1) : tid;

    // work item: block, share of planes, tile, neighbours next to each other on an XCD
    int w = xcd_run_order(blockIdx.x, gridDim.x);
    const int ti = w % C.tx; w /= C.tx;
    const int tj = w % C.ty; w /= C.ty;
    const int part = w % C.zs, lb = w/C.zs;
    const int nz = G.nc[2];
    const int k0 = (int)((long long)nz*part/C.zs), k1 = (int)((long long)nz*(part + 1)/C.zs);
    const int share = (nz + C.zs - 1)/C.zs;
    const int i0 = ti*C.wi, j0 = tj*C.wj;
    const int wi = min(C.wi, G.nc[0] - i0), wj = min(C.wj, G.nc[1] - j0);
    const TileLds Z(C.wi, C.wj, share, H, SS, MAP);
    const int PX = C.wi + 2*H, py = 3*PX;
    double* sS = lds + Z.sca;
    double* sFx = lds + Z.fx;
    double* sFy = lds + Z.fy;

    const bool active = tid < wi*wj;
    const int j = active ? tid/wi : 0, i = active ? tid - j*wi : 0;
    const int pos = (j + H)*PX + (i + H);
    const double ix = G.inv_dx[3*lb], iy = G.inv_dx[3*lb + 1], iz = G.inv_dx[3*lb + 2];

    // mapped coordinates: d x / d xi at the tile's cell centres (from -H) and
    // faces along each axis, with the per-cell code's map_deriv; when only y
    // is mapped (x and z derivatives 1.0 exactly) Jacobians and normals depend
    // on the row alone and are tabulated with the same expressions
    double* tX = lds + Z.tab;                 // centres x
    double* tY = tX + (C.wi + 2*H);           // centres y, Jacobian, normal (x, z faces), normal (y faces), 1/centre
    double* tZ = tY + 5*(C.wj + 2*H);         // centres z, from plane k0 - H
    double* fX = tZ + (share + Y);
    double* fY = fX + (C.wi + 1);             // faces y, normal at a y-face, 1/face
    double* fZ = fY + 3*(C.wj + 1);           // faces z, from plane k0
    const int nY = C.wj + 2*H, nYf = C.wj + 1;
    constexpr bool yonly = MAP == 1;
    if constexpr (MAP)
    {
        for (int t = tid; t < wi + 2*H; t += blockDim.x)
            tX[t] = map_deriv(G, 0, G.bmin[3*lb] + ((i0 + t - H) + 0.5)*G.dx[3*lb]);
        for (int t = tid; t <= wi; t += blockDim.x)
            fX[t] = map_deriv(G, 0, G.bmin[3*lb] + (((i0 + t) + 0.5) - 0.5)*G.dx[3*lb]);
        for (int t = tid; t < wj + 2*H; t += blockDim.x)
        {
            const double m = map_deriv(G, 1, G.bmin[3*lb + 1] + ((j0 + t - H) + 0.5)*G.dx[3*lb + 1]);
            const double jc = jac_at(1.0, m, 1.0);
            tY[t] = m; tY[nY + t] = jc; tY[2*nY + t] = nrm_at(1.0, jc); tY[3*nY + t] = nrm_at(m, jc); tY[4*nY + t] = 1.0/m;
        }
        for (int t = tid; t <= wj; t += blockDim.x)
        {
            const double m = map_deriv(G, 1, G.bmin[3*lb + 1] + (((j0 + t) + 0.5) - 0.5)*G.dx[3*lb + 1]);
            fY[t] = m; fY[nYf + t] = nrm_at(m, jac_at(1.0, m, 1.0)); fY[2*nYf + t] = 1.0/m;
        }
        for (int t = tid; t < k1 - k0 + 2*H; t += blockDim.x)
            tZ[t] = map_deriv(G, 2, G.bmin[3*lb + 2] + ((k0 + t - H) + 0.5)*G.dx[3*lb + 2]);
        for (int t = tid; t <= k1 - k0; t += blockDim.x)
            fZ[t] = map_deriv(G, 2, G.bmin[3*lb + 2] + (((k0 + t) + 0.5) - 0.5)*G.dx[3*lb + 2]);
    }

    // this thread's halo column: H layers beyond each side, and the corners
    // (the plan gives a tile at least as many threads as halo columns)
    const long long blk = (long long)lb*G.sb;
    const double* __restrict__ B = prims + blk;
    const int plane = G.nc[0]*G.N[1], xplane = G.N[1];
    const long long sv = G.sv;
    const int own = (int)stored_offset(G, i0 + i, j0 + j, 0);
    const int nhalo = 2*H*(wi + wj) + 4;
    int hpos = -1, hi = 0, hj = 0;
    const bool hcorner = rt >= nhalo - 4;
    if (rt < 2*H*wj)
    {
        const int a = rt/wj, lay = a >> 1;
        hj = rt - a*wj;
        hi = (a & 1) ? wi + lay : -1 - lay;
    }
    else if (rt < nhalo - 4)
    {
        const int t = rt - 2*H*wj, a = t/wi, lay = a >> 1;
        hi = t - a*wi;
        hj = (a & 1) ? wj + lay : -1 - lay;
    }
    else if (rt < nhalo)
    {
        const int c = rt - (nhalo - 4);
        hi = (c & 1) ? wi : -1; hj = (c & 2) ? wj : -1;
    }
    if (rt < nhalo) hpos = (hj + H)*PX + (hi + H);
    const int hoff = (int)stored_offset(G, i0 + hi, j0 + hj, 0);
    const int hstr = (i0 + hi >= 0 && i0 + hi < G.nc[0]) ? plane : xplane;
    auto load = [&](int off) -> Raw5
    {
        const double* e = B + off;
        return Raw5{e[0], e[sv], e[2*sv], e[3*sv], e[4*sv]};
    };
    auto put_vel = [&](double* s, int p, const Raw5& q) { s[3*p] = q.u; s[3*p + 1] = q.v; s[3*p + 2] = q.w; };
    auto put_sca = [&](int p, const TCell& c)
    {
        double* t = sS + SS*p;
        t[0] = c.p; t[1] = c.T;
        #pragma unroll
        for (int n = 0; n < S::extra; ++n) t[2 + n] = c.x[n];
    };
    auto cell_at_pos = [&](const double* s0, int p) -> TCell
    {
        const double* t = sS + SS*p;
        TCell c{t[0], t[1], s0[3*p], s0[3*p + 1], s0[3*p + 2], {0.0, 0.0, 0.0, 0.0}};
        #pragma unroll
        for (int n = 0; n < S::extra; ++n) c.x[n] = t[2 + n];
        return c;
    };

    // window of planes k0-1, k0, k0+1; plane k0+2 in flight
    double* rm = lds;
    double* rz = lds + Z.plane;
    double* rp = lds + 2*Z.plane;
    TCell cm{}, c0, c1;                       // own column at planes k-1 (wide), k, k+1
    Raw5 nr{}, hr{};                          // plane k+2 of the own and the halo column, as loaded
    double hp = 0.0, hT = 1.0;                // p, T of plane k+1 of the halo column (its velocities are in LDS)
    Raw5 below{};                             // own column at plane k0-2 (wide)
    const Raw5 q_m = load(own + (k0 - 1)*plane), q_0 = load(own + k0*plane), q_1 = load(own + (k0 + 1)*plane);
    if (S::wide) below = load(own + (k0 - 2)*plane);
    if (S::wide || k0 + 2 <= k1) nr = load(own + (k0 + 2)*plane);
    if (hpos >= 0)
    {
        const Raw5 a = load(hoff + (k0 - 1)*hstr), b = load(hoff + k0*hstr), c = load(hoff + (k0 + 1)*hstr);
        if (k0 + 2 <= k1) hr = load(hoff + (k0 + 2)*hstr);
        put_vel(rm, hpos, a); put_vel(rz, hpos, b); put_vel(rp, hpos, c);
        if (!hcorner) put_sca(hpos, derive<S>(C, b));
        hp = c.p; hT = c.T;
    }
    cm = derive<S>(C, q_m); c0 = derive<S>(C, q_0); c1 = derive<S>(C, q_1);
    if (active)
    {
        put_vel(rm, pos, q_m); put_vel(rz, pos, q_0); put_vel(rp, pos, q_1);
        put_sca(pos, c0);
    }
    lds_barrier();

    const double m0i = MAP ? tX[i + H] : 1.0, m1j = MAP ? tY[j + H] : 1.0;
    double zlo[5];
    // z-face between planes kf-1 and kf: normals of its cells and of the face
    auto z_normals = [&](int kf, double nc[NQ], double& nf, double& mf)
    {
        mf = fZ[kf - k0];
        if constexpr (yonly)
        {
            #pragma unroll
            for (int m = 0; m < NQ; ++m) nc[m] = tY[2*nY + j + H];
            nf = nc[0];
        }
        else
        {
            #pragma unroll
            for (int m = 0; m < NQ; ++m)
            {
                const double mz = tZ[kf - 1 - l + m - k0 + H];
                nc[m] = nrm_at(mz, jac_at(m0i, m1j, mz));
            }
            nf = nrm_at(mf, jac_at(m0i, m1j, mf));
        }
    };
    {
        double pw[1] = {1.0};
        if constexpr (S::power)
        {
            const double x[1] = {pow_arg(C, cm.T + c0.T)};
            pow_faces<1>(C.ps, x, C.power, false, pw);
        }
        double g[3][3] = {}, gT = 0.0, nc[NQ], nf = 1.0, mf = 1.0;
        #pragma unroll
        for (int m = 0; m < NQ; ++m) nc[m] = 1.0;
        if constexpr (MAP) z_normals(k0, nc, nf, mf);
        if constexpr (S::grad)
        {
            tile_grads_z<S>(rm, rz, py, 3*pos, cm, c0, ix, iy, iz, g, gT);
            if constexpr (yonly) grads_map_y<2>(g, gT, m1j, tY[4*nY + j + H]);
            else if constexpr (MAP) grads_map<2>(G, g, gT, mf, m0i, m1j);
        }
        if constexpr (S::wide)
        {
            const TCell q[4] = {derive<S>(C, below), cm, c0, c1};
            face_flux<2, S>(C, q, nc, nf, g, gT, zlo, pw[0]);
        }
        else
        {
            const TCell q[2] = {cm, c0};
            face_flux<2, S>(C, q, nc, nf, g, gT, zlo, pw[0]);
        }
        #pragma unroll
        for (int n = 0; n < 5; ++n) { if (!MAP) zlo[n] = zlo[n]*(sc*iz); }
    }

    // the closing faces of the tile are evaluated by lanes of the last two
    // waves, or all by the last one where it has no columns of its own
    const int nw = blockDim.x >> 6;
    const int by = rt - (nw - 1)*64;
    const int bx = wi*wj <= (nw - 1)*64 ? by : rt - max(nw - 2, 0)*64;

    const bool closing = __builtin_amdgcn_readfirstlane(rt) >= 64*max(nw - 2, 0);   // a wave with closing faces

    for (int k = k0; k < k1; ++k)
    {
        const Win W{rm, rz, rp, py};
        const double m2k = MAP ? tZ[k - k0 + H] : 1.0;
        const double jc = MAP ? (yonly ? tY[nY + j + H] : jac_at(m0i, m1j, m2k)) : 1.0;
        // the power law of the thread's three faces and of a closing face
        double pw[5] = {1.0, 1.0, 1.0, 1.0, 1.0};
        if constexpr (S::power)
        {
            const double* t = sS + 1;
            double x[5] = {1.0, 1.0, 1.0, 1.0, 1.0};
            if (active)
            {
                const double T0 = t[SS*pos];
                x[0] = pow_arg(C, t[SS*(pos - 1)] + T0);
                x[1] = pow_arg(C, t[SS*(pos - PX)] + T0);
                x[2] = pow_arg(C, T0 + c1.T);
            }
            if (bx >= 0 && bx < wj)
            {
                const int p = (bx + H)*PX + (wi + H);
                x[3] = pow_arg(C, t[SS*(p - 1)] + t[SS*p]);
            }
            if (by >= 0 && by < wi)
            {
                const int p = (wj + H)*PX + (by + H);
                x[4] = pow_arg(C, t[SS*(p - PX)] + t[SS*p]);
            }
            pow_faces<3>(C.ps, x, C.power, closing, pw);
        }
        double px[5], pyf[5], zhi[5], rin[5];
        const long long ro = blk + own + (long long)k*plane;
        TCell c2{};
        // x-face below cell ci (tile index) of row jj
        auto x_face = [&](int ci, int jj, int p, const TCell* mine, double pf, double P[5])
        {
            TCell q[NQ];
            #pragma unroll
            for (int m = 0; m < NQ; ++m)
                q[m] = (m == l + 1 && mine) ? *mine : cell_at_pos(rz, p - 1 - l + m);
            double g[3][3] = {}, gT = 0.0, nc[NQ], nf = 1.0;
            #pragma unroll
            for (int m = 0; m < NQ; ++m) nc[m] = 1.0;
            if constexpr (S::grad) tile_grads_x<S>(W, 3*(p - 1), q[l], q[l + 1], ix, iy, iz, g, gT);
            if constexpr (MAP)
            {
                const double m1 = tY[jj + H], mf = fX[ci];
                if constexpr (yonly)
                {
                    #pragma unroll
                    for (int m = 0; m < NQ; ++m) nc[m] = tY[2*nY + jj + H];
                    nf = nc[0];
                }
                else
                {
                    #pragma unroll
                    for (int m = 0; m < NQ; ++m)
                    {
                        const double mx = tX[ci - 1 - l + m + H];
                        nc[m] = nrm_at(mx, jac_at(mx, m1, m2k));
                    }
                    nf = nrm_at(mf, jac_at(mf, m1, m2k));
                }
                if constexpr (S::grad && yonly) grads_map_y<0>(g, gT, m1, tY[4*nY + jj + H]);
                else if constexpr (S::grad) grads_map<0>(G, g, gT, mf, m1, m2k);
            }
            face_flux<0, S>(C, q, nc, nf, g, gT, P, pf);
            #pragma unroll
            for (int n = 0; n < 5; ++n) { if (!MAP) P[n] = P[n]*(sc*ix); }
        };
        // y-face below cell (ii, cj)
        auto y_face = [&](int ii, int cj, int p, const TCell* mine, double pf, double P[5])
        {
            TCell q[NQ];
            #pragma unroll
            for (int m = 0; m < NQ; ++m)
                q[m] = (m == l + 1 && mine) ? *mine : cell_at_pos(rz, p + (m - 1 - l)*PX);
            double g[3][3] = {}, gT = 0.0, nc[NQ], nf = 1.0;
            #pragma unroll
            for (int m = 0; m < NQ; ++m) nc[m] = 1.0;
            if constexpr (S::grad) tile_grads_y<S>(W, 3*(p - PX), q[l], q[l + 1], ix, iy, iz, g, gT);
            if constexpr (MAP)
            {
                const double m0 = tX[ii + H], mf = fY[cj];
                if constexpr (yonly)
                {
                    #pragma unroll
                    for (int m = 0; m < NQ; ++m) nc[m] = tY[3*nY + cj - 1 - l + m + H];
                    nf = fY[nYf + cj];
                }
                else
                {
                    #pragma unroll
                    for (int m = 0; m < NQ; ++m)
                    {
                        const double my = tY[cj - 1 - l + m + H];
                        nc[m] = nrm_at(my, jac_at(m0, my, m2k));
                    }
                    nf = nrm_at(mf, jac_at(m0, mf, m2k));
                }
                if constexpr (S::grad && yonly) grads_map_y<1>(g, gT, mf, fY[2*nYf + cj]);
                else if constexpr (S::grad) grads_map<1>(G, g, gT, mf, m2k, m0);
            }
            face_flux<1, S>(C, q, nc, nf, g, gT, P, pf);
            #pragma unroll
            for (int n = 0; n < 5; ++n) { if (!MAP) P[n] = P[n]*(sc*iy); }
        };
        // the sections below are kept apart (sched_barrier): interleaved, the
        // wide compositions' faces need more registers than there are.  Wide:
        // the own cell of plane k and the own low faces are read from LDS where
        // used, and the z-face, with its plane k+2, comes last
        if (active)
        {
            x_face(i, j, pos, S::wide ? nullptr : &c0, pw[0], px);
            #pragma unroll
            for (int n = 0; n < 5; ++n) sFx[(j*(C.wi + 1) + i)*5 + n] = px[n];
            if constexpr (S::wide) __builtin_amdgcn_sched_barrier(0);
            y_face(i, j, pos, S::wide ? nullptr : &c0, pw[1], pyf);
            #pragma unroll
            for (int n = 0; n < 5; ++n) sFy[(j*C.wi + i)*5 + n] = pyf[n];
            if constexpr (S::wide) __builtin_amdgcn_sched_barrier(0);
        }
        if (bx >= 0 && bx < wj)
        {
            double P[5];
            x_face(wi, bx, (bx + H)*PX + (wi + H), nullptr, pw[3], P);
            #pragma unroll
            for (int n = 0; n < 5; ++n) sFx[(bx*(C.wi + 1) + wi)*5 + n] = P[n];
        }
        if (by >= 0 && by < wi)
        {
            double P[5];
            y_face(by, wj, (wj + H)*PX + (by + H), nullptr, pw[4], P);
            #pragma unroll
            for (int n = 0; n < 5; ++n) sFy[(wj*C.wi + by)*5 + n] = P[n];
        }
        if (active)
        {
            if constexpr (S::wide)
            {
                __builtin_amdgcn_sched_barrier(0);
                c0 = cell_at_pos(rz, pos);
                c2 = derive<S>(C, nr);
            }
            double g[3][3] = {}, gT = 0.0, nc[NQ], nf = 1.0, mf = 1.0;
            #pragma unroll
            for (int m = 0; m < NQ; ++m) nc[m] = 1.0;
            if constexpr (MAP) z_normals(k + 1, nc, nf, mf);
            if constexpr (S::grad)
            {
                tile_grads_z<S>(rz, rp, py, 3*pos, c0, c1, ix, iy, iz, g, gT);
                if constexpr (yonly) grads_map_y<2>(g, gT, m1j, tY[4*nY + j + H]);
            else if constexpr (MAP) grads_map<2>(G, g, gT, mf, m0i, m1j);
            }
            if constexpr (S::wide)
            {
                const TCell q[4] = {cm, c0, c1, c2};
                face_flux<2, S>(C, q, nc, nf, g, gT, zhi, pw[2]);
            }
            else
            {
                const TCell q[2] = {c0, c1};
                face_flux<2, S>(C, q, nc, nf, g, gT, zhi, pw[2]);
            }
            #pragma unroll
            for (int n = 0; n < 5; ++n) { if (!MAP) zhi[n] = zhi[n]*(sc*iz); keep_here(zhi[n]); }
        }
        // increment mode: requested before the barrier, so that the wait for
        // the other waves covers its latency
        #pragma unroll
        for (int n = 0; n < 5; ++n) rin[n] = increment && active ? rhs[ro + n*sv] : 0.0;
        lds_barrier();
        if (active)
        {
            // faces in the order x-, x+, y-, y+, z-, z+ (flux_div_basic.h:54-72)
            #pragma unroll
            for (int n = 0; n < 5; ++n)
            {
                double r = rin[n];
                const double xh = sFx[(j*(C.wi + 1) + i + 1)*5 + n], yh = sFy[((j + 1)*C.wi + i)*5 + n];
                const double xl = S::wide ? sFx[(j*(C.wi + 1) + i)*5 + n] : px[n];
                const double yl = S::wide ? sFy[(j*C.wi + i)*5 + n] : pyf[n];
                if constexpr (MAP)
                {
                    const double fx = sc*(jc*ix), fy = sc*(jc*iy), fz = sc*(jc*iz);
                    r += xl*fx; r -= xh*fx;
                    r += yl*fy; r -= yh*fy;
                    r += zlo[n]*fz; r -= zhi[n]*fz;
                }
                else
                {
                    r += xl;     r -= xh;
                    r += yl;     r -= yh;
                    r += zlo[n]; r -= zhi[n];
                }
                rhs[ro + n*sv] = r;
                zlo[n] = zhi[n];
            }
        }
        if (k + 1 < k1)
        {
            // plane k+2 takes the slot of plane k-1; the scalars move to plane k+1
            double* t = rm; rm = rz; rz = rp; rp = t;
            if (active)
            {
                put_sca(pos, c1);
                if constexpr (S::wide) { rp[3*pos] = c2.u; rp[3*pos + 1] = c2.v; rp[3*pos + 2] = c2.w; }
                else put_vel(rp, pos, nr);
            }
            cm = c0; c0 = c1;
            if constexpr (S::wide)
            {
                c1 = c2;
                if (k + 3 <= k1 + 1) nr = load(own + (k + 3)*plane);
            }
            else
            {
                c1 = derive<S>(C, nr);
                if (k + 3 <= k1) nr = load(own + (k + 3)*plane);
            }
            if (hpos >= 0)
            {
                if (!hcorner)
                    put_sca(hpos, derive<S>(C, Raw5{hp, hT, rz[3*hpos], rz[3*hpos + 1], rz[3*hpos + 2]}));
                put_vel(rp, hpos, hr);
                hp = hr.p; hT = hr.T;
                if (k + 3 <= k1) hr = load(hoff + (k + 3)*hstr);
            }
        }
        lds_barrier();
    }
}

// The tiling of a launch: columns per tile so that a tile has at most 256
// columns (and 64 along each side, the lanes of a closing-face wave), picked
// by what its workgroups cost -- waves, counting idle lanes, plus a quarter of
// a thread per halo column it loads again and the two closing-face passes (a
// third of a wave's faces each) -- and workgroups along k by rounds
// of resident workgroups (as fast_zsplit), a share costing its planes plus
// kTilePrologue for its prologue: twelve 4 x 8 x 4 blocks run as 24 workgroups, 27
// blocks of 32^3 as 432, 240 blocks of 24 x 20 x 12 as 480 of half a block each.
//
// The search runs on every call, so it steps from one tile side (and one share
// of planes) to the next smaller one and not through every count of tiles,
// most of which leave the side as it is: some hundred candidates for any
// block.  One by one, a 512 x 512 x 2 block cost 226 us of host time a call, more than
// three times what its {KEEP2} residual takes, and a 2048 x 2048 x 2 one 3500 us.
constexpr double kTilePrologue = 0.65;
struct TilePlan { int wi, wj, tx, ty, zs, nt; size_t lds; };

inline int ceil_div(int a, int b) { return (a + b - 1)/b; }

// the least number of parts of n that makes the largest smaller than part (n + 1: none does)
inline int parts_below(int n, int part) { return part > 1 ? ceil_div(n, part - 1) : n + 1; }

// threads of a tile's workgroup
inline int tile_threads(int H, int wi, int wj) { return 64*ceil_div(std::max(wi*wj, 2*H*(wi + wj) + 4), 64); }

// cost of the tiles of a cross-section in threads, infinite where a tile has too many
inline double tile_cost(const DevGeom& G, int H, int wi, int wj)
{
    const int nt = tile_threads(H, wi, wj);
    if (nt > 256) return 1e300;
    return (double)ceil_div(G.nc[0], wi)*ceil_div(G.nc[1], wj)*(nt + 0.25*(2*H*(wi + wj) + 4) + 128.0/3.0);
}

// cost of a tiling's planes shared out to zs workgroups
inline double share_cost(const DevGeom& G, const TilePlan& p, int zs, size_t lds, int cus)
{
    const int per_cu = std::max(1, std::min((int)(160*1024/(lds + 2048)), 512/p.nt));
    const double rounds = std::ceil((double)p.tx*p.ty*G.nblk*zs/((double)per_cu*cus));
    return rounds*(ceil_div(G.nc[2], zs) + kTilePrologue);
}

inline TilePlan plan_tile(const DevGeom& G, int H, int SS, bool map, int cus)
{
    TilePlan best{};
    double best_cost = 1e299;
    const int nx = G.nc[0], ny = G.nc[1], nz = G.nc[2];
    for (int tx = ceil_div(nx, 64), wi; tx <= ceil_div(nx, 4); tx = parts_below(nx, wi))
    {
        wi = ceil_div(nx, tx);
        for (int ty = ceil_div(ny, std::min(64, 256/wi)), wj; ty <= ny; ty = parts_below(ny, wj))
        {
            wj = ceil_div(ny, ty);
            const double cost = tile_cost(G, H, wi, wj);
            if (cost < best_cost - 1e-9)
            {
                best_cost = cost;
                best = TilePlan{wi, wj, ceil_div(nx, wi), ceil_div(ny, wj), 1, tile_threads(H, wi, wj), 0};
            }
        }
    }
    best_cost = 1e300;
    for (int zs = ceil_div(nz, 64), share; zs <= nz; zs = parts_below(nz, share))
    {
        share = ceil_div(nz, zs);
        const size_t lds = sizeof(double)*(size_t)TileLds(best.wi, best.wj, share, H, SS, map).total;
        const double cost = share_cost(G, best, zs, lds, cus);
        if (cost < best_cost - 1e-9) { best_cost = cost; best.zs = zs; best.lds = lds; }
    }
    return best;
}

inline TileCfg tile_cfg(const spd_flux_desc& f, double scale)
{
    TileCfg C{};
    cfg_gas(C, f);
    C.scale = scale;
    C.gamma = f.gamma;
    C.gamma_R = f.gamma*f.R;
    for (int m = 0; m < f.nterms; ++m)
    {
        const spd_flux_term& t = f.terms[m];
        if (t.kind == SPD_TERM_PDISS) cfg_pdiss(C, t, scale);
        else if (t.kind == SPD_TERM_VISC)
        {
            cfg_visc(C, t, scale);
            C.alpha_s = scale*(t.mu*(1.0/t.prandtl));
            C.sgs_cw = t.sgs_cw; C.sgs_delta = t.sgs_delta; C.sgs_prt = t.sgs_prt;
        }
        else { C.split_phys = t.split == SPD_SPLIT_PHYS; C.smooth = t.smooth; }
    }
    return C;
}

template <class S>
void launch_tile(const Grid& g, const double* prims, double* rhs, const spd_flux_desc& f, bool increment,
                 hipStream_t s, int cus)
{
    const DevGeom& G = g.geom;
    const bool map = !G.identity;
    const TilePlan p = plan_tile(G, S::H, S::SS, map, cus);
    TileCfg C = tile_cfg(f, S::scale);
    C.wi = p.wi; C.wj = p.wj; C.tx = p.tx; C.ty = p.ty; C.zs = p.zs;
    const dim3 grid((unsigned)(p.tx*p.ty*p.zs*G.nblk)), block((unsigned)p.nt);
    const int inc = increment ? 1 : 0;
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, p.lds, s, G, prims, rhs, C, inc); };
    switch (map_variant(G))
    {
        case 0: go(k_flux_div_spec_tile<S, 0>); break;
        case 1: go(k_flux_div_spec_tile<S, 1>); break;
        case 2: go(k_flux_div_spec_tile<S, 2>); break;
    }
    SPD_LAUNCH_CHECK();
}

// the viscous part of a composition: 0 none, 1 + law, + 2 with WALE
inline int visc_variant(const spd_flux_desc& f)
{
    for (int m = 0; m < f.nterms; ++m)
        if (f.terms[m].kind == SPD_TERM_VISC) return 1 + f.terms[m].law + (f.terms[m].sgs == SPD_SGS_WALE ? 2 : 0);
    return 0;
}

template <int CONV, int PDISS>
bool tile_visc(const Grid& g, const double* prims, double* rhs, const spd_flux_desc& f, bool inc, hipStream_t s,
               int cus)
{
    switch (visc_variant(f))
    {
        case 0:
            if constexpr (CONV != CV_NONE || PDISS != 0)
            {
                launch_tile<TileSpec<CONV, PDISS, 0>>(g, prims, rhs, f, inc, s, cus);
                return true;
            }
            return false;
        case 1: launch_tile<TileSpec<CONV, PDISS, 1>>(g, prims, rhs, f, inc, s, cus); return true;
        case 2: launch_tile<TileSpec<CONV, PDISS, 2>>(g, prims, rhs, f, inc, s, cus); return true;
        case 3: launch_tile<TileSpec<CONV, PDISS, 3>>(g, prims, rhs, f, inc, s, cus); return true;
        case 4: launch_tile<TileSpec<CONV, PDISS, 4>>(g, prims, rhs, f, inc, s, cus); return true;
    }
    return false;
}

} // namespace
} // namespace spd
