// Generic flux_div: one thread per interior cell, six face evaluations per
// cell in the order of the reference's flux_div_basic
// (pde-algs/flux-div/flux_div_basic.h:47-72): for idir in 0..2, pm in 0..1,
// accum = F(face); accum *= jac*(1-2pm)*inv_dx; rhs += accum.
//
// k_flux_div_generic dispatches the terms at run time and serves every
// composition the library supports.  The compositions with compile-time code
// (flux_div_spec_code) run face-once kernels instead: the 16 x 16 kernel of
// flux_fast.hip for cent_keep<2>, pressure_diss_lr and visc_lr on blocks of that
// cross-section, the tiled kernel of flux_tile.hpp for everything else.
// Compiled without floating-point contraction and in the reference's
// expression order, so for identity coordinates a result equals the reference
// bit for bit except where a libm routine (pow, tanh) is involved.
#include "spd_internal.hpp"
#include "flux_cell.hpp"
#include <cmath>
#include <algorithm>

namespace spd {
namespace {

// The run-time term dispatch of the generic kernel.  SPD_TERM_HYBRID has no
// device code: validate_flux refuses it before any launch.  FWENO: built with
// fweno_t, whose unrolled arrays are worth 1 to 20 % to compositions with it
// (24x20x12 blocks, {KEEP2, FWENO}: 413 -> 341 us) but spill 79 registers instead of
// 26, which cost the others 2 to 7 % ({pressure diffusion, Totani} 379 -> 405 us).
template <bool FWENO>
__device__ __forceinline__ void eval_term(const Cell& C, const FaceIdx& f, const spd_flux_term& t, double R, double gam, double out[5])
{
    switch (t.kind)
    {
        case SPD_TERM_KEEP:   f_keep(C, f, t.order, R, gam, out); break;
        case SPD_TERM_TOTANI: f_totani(C, f, R, gam, out); break;
        case SPD_TERM_PDISS:  f_pdiss(C, f, t, R, gam, out); break;
        case SPD_TERM_WENO:   f_weno(C, f, t, R, gam, out); break;
        case SPD_TERM_FIRST:  f_first(C, f, R, gam, out); break;
        case SPD_TERM_VISC:   f_visc(C, f, t, R, gam, out); break;
        case SPD_TERM_WENO_FDS: f_weno_fds(C, f, t, R, gam, out); break;
        default:
            if constexpr (FWENO) if (t.kind == SPD_TERM_FWENO) { f_fweno(C, f, t, R, gam, out); break; }
            for (int n = 0; n < 5; ++n) out[n] = 0.0;
    }
}

// rhs of cell (i, j, k) of block lb in the reference's per-cell order
// (flux_div_basic.h:47-72)
template <bool FWENO>
__device__ inline void generic_cell(const DevGeom& G, const double* __restrict__ prims, double* __restrict__ rhs,
                                    const spd_flux_desc& F, const PowAt& ps, int increment, int i, int j, int k, int lb)
{
    Cell C{&G, prims + (long long)lb*G.sb, lb, &ps};
    double jac = 1.0;
    if (!G.identity)
    {
        double xi[3]; cell_xi(G, lb, i, j, k, xi);
        jac = 1.0/(map_deriv(G, 0, xi[0])*map_deriv(G, 1, xi[1])*map_deriv(G, 2, xi[2]));
    }
    double relem[5];
    for (int v = 0; v < 5; ++v) relem[v] = increment ? rhs[cell_index(G, lb, v, i, j, k)] : 0.0;
    for (int idir = 0; idir < 3; ++idir)
    {
        const double inv_dx = 1.0/G.dx[3*lb + idir];
        for (int pm = 0; pm < 2; ++pm)
        {
            FaceIdx f{idir, i, j, k};
            if (pm == 1) { if (idir == 0) f.i++; else if (idir == 1) f.j++; else f.k++; }
            // compose: F0 + (F1 + (... + Fn))
            double acc[5];
            eval_term<FWENO>(C, f, F.terms[F.nterms - 1], F.R, F.gamma, acc);
            for (int m = F.nterms - 2; m >= 0; --m)
            {
                double z[5];
                eval_term<FWENO>(C, f, F.terms[m], F.R, F.gamma, z);
                for (int n = 0; n < 5; ++n) { z[n] += acc[n]; acc[n] = z[n]; }
            }
            const double s = jac*(1.0 - 2.0*pm)*inv_dx;
            for (int n = 0; n < 5; ++n) { acc[n] *= s; relem[n] += acc[n]; }
        }
    }
    for (int v = 0; v < 5; ++v) rhs[cell_index(G, lb, v, i, j, k)] = relem[v];
}

template <bool FWENO>
__global__ void __launch_bounds__(256) __attribute__((flatten))
k_flux_div_generic(DevGeom G, const double* __restrict__ prims, double* __restrict__ rhs, spd_flux_desc F, PowAt ps,
                   int increment)
{
    const int tiles_x = (G.nc[0] + 15)/16, tiles_y = (G.nc[1] + 15)/16;
    long long w = blockIdx.x;
    const int tx = (int)(w % tiles_x); w /= tiles_x;
    const int ty = (int)(w % tiles_y); w /= tiles_y;
    const int k  = (int)(w % G.nc[2]); w /= G.nc[2];
    const int lb = (int)w;
    const int i = tx*16 + (threadIdx.x & 15);
    const int j = ty*16 + (threadIdx.x >> 4);
    // geometry and flux descriptor in LDS: the per-cell code indexes them
    // with run-time values, which on kernel arguments would make every lane
    // copy them to private (scratch) memory first
    __shared__ DevGeom sG;
    __shared__ spd_flux_desc sF;
    __shared__ PowAt sP;
    if (threadIdx.x == 0) { sG = G; sF = F; sP = ps; }
    __syncthreads();
    if (i >= G.nc[0] || j >= G.nc[1]) return;
    generic_cell<FWENO>(sG, prims, rhs, sF, sP, increment, i, j, k, lb);
}

} // namespace

// Compositions with compile-time code, as term codes T0 T1 T2 (0: none)
#define SPD_SPEC_LIST(X) \
    X(SPD_TERM_KEEP, 0, 0) X(SPD_TERM_PDISS, 0, 0) X(SPD_TERM_KEEP, SPD_TERM_PDISS, 0) \
    X(SPD_TERM_VISC, 0, 0) X(SPD_TERM_KEEP, SPD_TERM_VISC, 0) X(SPD_TERM_PDISS, SPD_TERM_VISC, 0) \
    X(SPD_TERM_KEEP, SPD_TERM_PDISS, SPD_TERM_VISC) \
    X(TERM_KEEP4, 0, 0) X(SPD_TERM_TOTANI, 0, 0) X(SPD_TERM_WENO, 0, 0) X(SPD_TERM_FWENO, 0, 0) \
    X(SPD_TERM_FIRST, 0, 0) X(TERM_KEEP4, SPD_TERM_VISC, 0) X(SPD_TERM_TOTANI, SPD_TERM_VISC, 0) \
    X(SPD_TERM_WENO, SPD_TERM_VISC, 0) X(SPD_TERM_FWENO, SPD_TERM_VISC, 0) X(SPD_TERM_FIRST, SPD_TERM_VISC, 0) \
    X(SPD_TERM_WENO_FDS, 0, 0) X(SPD_TERM_WENO_FDS, SPD_TERM_VISC, 0)

bool flux_has_hybrid(const spd_flux_desc& f)
{
    for (int m = 0; m < f.nterms && m < SPD_MAX_TERMS; ++m) if (f.terms[m].kind == SPD_TERM_HYBRID) return true;
    return false;
}

int flux_div_spec_code(const spd_flux_desc& f)
{
    // SPD_DISABLE_SPEC=1 sends every composition to the generic kernel (for
    // timing comparisons)
    if (const char* e = getenv("SPD_DISABLE_SPEC")) if (e[0] == '1') return 0;
    if (f.nterms < 1 || f.nterms > 3) return 0;
    int code = 0;
    for (int m = 0; m < f.nterms; ++m)
    {
        const spd_flux_term& t = f.terms[m];
        int k = t.kind;
        if (k == SPD_TERM_KEEP) { if (t.order == 4) k = TERM_KEEP4; else if (t.order != 2) return 0; }
        else if ((k < SPD_TERM_TOTANI || k > SPD_TERM_VISC) && k != SPD_TERM_WENO_FDS) return 0;
        code = code*100 + k;
    }
    for (int m = f.nterms; m < 3; ++m) code *= 100;
#define SPD_SPEC_MATCH(a, b, c) if (code == (a)*10000 + (b)*100 + (c)) return code;
    SPD_SPEC_LIST(SPD_SPEC_MATCH)
#undef SPD_SPEC_MATCH
    return 0;
}

// the tiled kernel's translation units (flux_tile_*.hip): false when the pair
// (convective term code, 1 + pressure-diffusion sensor) is not theirs
#define SPD_TILE_DECL(name) \
    bool name(const Grid& g, const double* prims, double* rhs, const spd_flux_desc& f, int conv, int pdiss, bool inc, \
              hipStream_t s, int cus);
SPD_TILE_DECL(tile_central) SPD_TILE_DECL(tile_pdiss) SPD_TILE_DECL(tile_split) SPD_TILE_DECL(tile_weno)
#undef SPD_TILE_DECL

bool launch_flux_div_tile(const Grid& g, const double* prims, double* rhs, const spd_flux_desc& f, bool increment,
                          hipStream_t s)
{
    if (!flux_div_spec_code(f) || !tile_offsets_fit(g.geom)) return false;
    int conv = CV_NONE, pdiss = 0;
    for (int m = 0; m < f.nterms; ++m)
        switch (f.terms[m].kind)
        {
            case SPD_TERM_KEEP:     conv = f.terms[m].order == 4 ? CV_KEEP4 : CV_KEEP2; break;
            case SPD_TERM_TOTANI:   conv = CV_TOTANI; break;
            case SPD_TERM_WENO:     conv = CV_WENO; break;
            case SPD_TERM_FWENO:    conv = CV_FWENO; break;
            case SPD_TERM_FIRST:    conv = CV_FIRST; break;
            case SPD_TERM_WENO_FDS: conv = CV_FDS; break;
            case SPD_TERM_PDISS:    pdiss = 1 + f.terms[m].sensor; break;
            default: break;
        }
    const int cus = g.ctx->cus;
    return tile_central(g, prims, rhs, f, conv, pdiss, increment, s, cus)
        || tile_pdiss(g, prims, rhs, f, conv, pdiss, increment, s, cus)
        || tile_split(g, prims, rhs, f, conv, pdiss, increment, s, cus)
        || tile_weno(g, prims, rhs, f, conv, pdiss, increment, s, cus);
}

void launch_flux_div_generic(const Grid& g, const double* prims, double* rhs, const spd_flux_desc& f,
                             bool increment, hipStream_t s)
{
    // compositions with compile-time code run tiled; any other one through the
    // run-time term dispatch, one thread per cell
    if (launch_flux_div_tile(g, prims, rhs, f, increment, s)) return;
    const DevGeom& G = g.geom;
    const long long nwg = (long long)((G.nc[0] + 15)/16)*((G.nc[1] + 15)/16)*G.nc[2]*G.nblk;
    bool fweno = false;
    for (int m = 0; m < f.nterms; ++m) fweno |= f.terms[m].kind == SPD_TERM_FWENO;
    auto kernel = fweno ? k_flux_div_generic<true> : k_flux_div_generic<false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)nwg), dim3(256), 0, s, G, prims, rhs, f, pow_of(f), increment ? 1 : 0);
    SPD_LAUNCH_CHECK();
}

} // namespace spd
