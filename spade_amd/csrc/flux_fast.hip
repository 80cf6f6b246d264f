// LDS-staged flux_div for the hot combinations on gfx950:
//   cent_keep<2> [+ pressure_diss_lr (const | Ducros)] [+ visc_lr (const | power law)]
// on identity or diagonal (tanh) coordinates and blocks with a 16x16 (i,j)
// cross-section.
//
// One workgroup (256 threads, thread (i,j)) owns a block, or a share of its
// planes, and marches over k.
// Every face flux is evaluated once: thread (i,j) evaluates the low x-face
// i-1/2, the low y-face j-1/2 and the high z-face k+1/2 of its cell; the 16
// block-boundary x-faces and the 16 y-faces of a plane are evaluated by 16
// lanes of waves 2 and 3.  In-plane face products P = F * (1/dx) are exchanged
// through LDS; the z-face product stays in registers for the next plane.
//
// LDS holds, for the three planes k-1, k, k+1, the velocities (u,v,w) on the
// 18x18 plane with one halo layer (ring of three slots), and for planes k and
// k+1 the p, T, rho, e needed as left/right states of the faces.
//
// Power law: x^n comes from a binomial series valid near x = 1, and from the
// library pow for faces outside its range (pow_faces).
//
// Arithmetic follows the reference's expression order exactly
// (navier-stokes/convective.h:117-184, 212-245; viscous.h:39-112;
// omni/infos/info_gradient.h:45-81; pde-algs/flux-div/flux_div_basic.h:47-72)
// and the file is compiled without contraction, so the result equals the
// reference bit for bit except through pow() of the power-law viscosity
// (a binomial series within one ulp of x^n, see pow_series.hpp).
// Per-cell quantities the reference recomputes for every face (rho = p/(R T),
// e = p/(rho (gamma-1))) are computed once per cell: same operands, same
// rounding.
#include "spd_internal.hpp"
#include "flux_face.hpp"
#include "spd_stage.hpp"
#include <algorithm>
#include <cstdlib>

namespace spd {
namespace {

constexpr int HX = 18, HP = 18*18;


// slot s of the velocity ring: s[pos] = u, s[HP + pos] = v, s[2*HP + pos] = w

template <class S>
__device__ inline void grads_x(const double* sm, const double* s0, const double* sp, int pL, int pR,
                               const CellV& L, const CellV& R, double ix, double iy, double iz,
                               double g[3][3], double& gT)
{
    g[0][0] = normal_grad(L.u, R.u, ix);
    g[0][1] = normal_grad(L.v, R.v, ix);
    g[0][2] = normal_grad(L.w, R.w, ix);
    gT      = normal_grad(L.T, R.T, ix);
    g[1][0] = tang(s0[pL + HX], s0[pL - HX], s0[pR + HX], s0[pR - HX], iy);
    g[1][1] = tang(s0[HP + pL + HX], s0[HP + pL - HX], s0[HP + pR + HX], s0[HP + pR - HX], iy);
    g[1][2] = S::full_grad ? tang(s0[2*HP + pL + HX], s0[2*HP + pL - HX], s0[2*HP + pR + HX], s0[2*HP + pR - HX], iy) : 0.0;
    g[2][0] = tang(sp[pL], sm[pL], sp[pR], sm[pR], iz);
    g[2][1] = S::full_grad ? tang(sp[HP + pL], sm[HP + pL], sp[HP + pR], sm[HP + pR], iz) : 0.0;
    g[2][2] = tang(sp[2*HP + pL], sm[2*HP + pL], sp[2*HP + pR], sm[2*HP + pR], iz);
}

template <class S>
__device__ inline void grads_y(const double* sm, const double* s0, const double* sp, int pL, int pR,
                               const CellV& L, const CellV& R, double ix, double iy, double iz,
                               double g[3][3], double& gT)
{
    g[1][0] = normal_grad(L.u, R.u, iy);
    g[1][1] = normal_grad(L.v, R.v, iy);
    g[1][2] = normal_grad(L.w, R.w, iy);
    gT      = normal_grad(L.T, R.T, iy);
    g[2][0] = S::full_grad ? tang(sp[pL], sm[pL], sp[pR], sm[pR], iz) : 0.0;
    g[2][1] = tang(sp[HP + pL], sm[HP + pL], sp[HP + pR], sm[HP + pR], iz);
    g[2][2] = tang(sp[2*HP + pL], sm[2*HP + pL], sp[2*HP + pR], sm[2*HP + pR], iz);
    g[0][0] = tang(s0[pL + 1], s0[pL - 1], s0[pR + 1], s0[pR - 1], ix);
    g[0][1] = tang(s0[HP + pL + 1], s0[HP + pL - 1], s0[HP + pR + 1], s0[HP + pR - 1], ix);
    g[0][2] = S::full_grad ? tang(s0[2*HP + pL + 1], s0[2*HP + pL - 1], s0[2*HP + pR + 1], s0[2*HP + pR - 1], ix) : 0.0;
}

template <class S>
__device__ inline void grads_z(const double* sL, const double* sR, int p,
                               const CellV& L, const CellV& R, double ix, double iy, double iz,
                               double g[3][3], double& gT)
{
    g[2][0] = normal_grad(L.u, R.u, iz);
    g[2][1] = normal_grad(L.v, R.v, iz);
    g[2][2] = normal_grad(L.w, R.w, iz);
    gT      = normal_grad(L.T, R.T, iz);
    g[0][0] = tang(sL[p + 1], sL[p - 1], sR[p + 1], sR[p - 1], ix);
    g[0][1] = S::full_grad ? tang(sL[HP + p + 1], sL[HP + p - 1], sR[HP + p + 1], sR[HP + p - 1], ix) : 0.0;
    g[0][2] = tang(sL[2*HP + p + 1], sL[2*HP + p - 1], sR[2*HP + p + 1], sR[2*HP + p - 1], ix);
    g[1][0] = S::full_grad ? tang(sL[p + HX], sL[p - HX], sR[p + HX], sR[p - HX], iy) : 0.0;
    g[1][1] = tang(sL[HP + p + HX], sL[HP + p - HX], sR[HP + p + HX], sR[HP + p - HX], iy);
    g[1][2] = tang(sL[2*HP + p + HX], sL[2*HP + p - HX], sR[2*HP + p + HX], sR[2*HP + p - HX], iy);
}

__device__ inline CellV cell_from_lds(const double* sS, const double* s0, int p)
{
    // sS: [p, T, rho, e][HP] of plane k; s0: ring slot of plane k
    return CellV{sS[p], sS[HP + p], s0[p], s0[HP + p], s0[2*HP + p], sS[2*HP + p], sS[3*HP + p]};
}

__device__ inline int lpos(int i, int j) { return (j + 1)*HX + (i + 1); }

struct Raw { double p, T, u, v, w; };

// The RK stage a fused launch applies to each cell once its residual L is
// known (transform-aware, time-integration/advance.h:56-102):
//   qout = c2p(p2c(q) + c[0] r[0] + .. + c[n-2] r[n-2] + c[n-1] L)
// in k_rk_transform's order (nonzero coefficients only), then pushed into the
// ghosts of qout it feeds.
struct StageArgs
{
    double* qout;
    const double* r[2];          // residuals of the earlier stages, rhs layout
    double c[3];
    int n;                       // 1..3 coefficients, the last one for L
    int store_rhs;               // also write L to rhs
    double gamma, R, inv_gm1;    // inv_gm1 = 1/(gamma - 1)
    int same_R;                  // R is the flux's gas constant
    const int* push;             // push table (d_push)
    int push_ghosts;             // write the ghosts this stage's result feeds
    const int* nbr;              // source table (d_nbr), read halos from neighbour interiors (STG == 2)
    double t_wall;               // isothermal wall temperature (wall_y)
    int wall_y;                  // STG == 2: y faces without a source block are isothermal walls
};

// STG: 0 flux_div only; 1 fused stage, halo from this block's ghost cells;
// 2 fused stage, halo from the neighbour blocks' interiors (every ghost
// region has a source block, or, in the mapped kernel, the y regions without
// one are isothermal walls whose ghosts are formed from the mirrored cells)
// MAP: 0 identity coordinates, 1 only y mapped, 2 any diagonal map
template <int KEEP, int PDISS, int VISC, bool INC, int MAP, int STG = 0>
__global__ void __launch_bounds__(256, 2)
k_flux_fast(DevGeom G, const double* __restrict__ prims, double* __restrict__ rhs, FastCfg C, StageArgs A, int split)
{
    using S = Spec<KEEP, PDISS, VISC>;
    static_assert(!(STG && INC), "a fused stage writes a fresh residual");
    // x-ghost pushes of a fused stage: the plane's cells within ng of an x
    // face, staged for whole-row writes (flushed after the next barrier)
    __shared__ double sXs[STG ? sizeof(XStage)/sizeof(double) : 1];
    XStage& xs = *reinterpret_cast<XStage*>(sXs);
    // mapped coordinates: d x_a / d xi_a of this block at cell centres -1 .. 16
    // and at faces 0 .. 16 of each axis, from the same map_deriv as the
    // per-cell kernels (so the same bits)
    __shared__ double sMc[MAP ? 3 : 1][18], sMf[MAP ? 3 : 1][17];
    // mapped y only (x and z identity, so their d x / d xi are 1.0 exactly):
    // every face normal and Jacobian depends on the row alone, tabulated per
    // block with the same expressions: sY[0][r] = jac at cell row r - 1,
    // sY[1][r] = its normal factor 1/(1 jac), sY[2][r] = the y-face normal
    // factor of a cell row, sY[3][f] = the y-face normal factor at face f,
    // sY[4][r] and sY[5][f] = 1/(d y / d eta) there
    __shared__ double sY[MAP == 1 ? 6 : 1][18];
    __shared__ double sU[3][3*HP];        // u, v, w of planes k-1, k, k+1 (ring)
    __shared__ double sS[2][4*HP];        // p, T, rho, e of planes k, k+1 (by parity)
    __shared__ double sFx[5][16*17];      // x-face products, faces i = 0..16 of row j
    __shared__ double sFy[5][17*16];      // y-face products, faces j = 0..16 of column i

    // zsplit workgroups per block, each marching over its share of the planes
    // [k0, k1) with its own window prologue: small grids fill the device, and the
    // tail rounds of a middling one are shorter
    // split: workgroups per block in the low byte, bit 8 set for XCD runs
    const int zsplit = split & 0xff;
    const int w = (split & 0x100) ? xcd_run_order(blockIdx.x, G.nblk*zsplit) : blockIdx.x;
    const int lb = w/zsplit, half = w - lb*zsplit;
    const int k0 = G.nc[2]*half/zsplit, k1 = G.nc[2]*(half + 1)/zsplit;
    const int tid = threadIdx.x;
    const int i = tid & 15, j = tid >> 4;
    const double ix = G.inv_dx[3*lb + 0], iy = G.inv_dx[3*lb + 1], iz = G.inv_dx[3*lb + 2];
    constexpr bool yonly = MAP == 1;
    if constexpr (MAP)
    {
        if (tid < 54)
        {
            const int a = tid/18, c = tid % 18 - 1;
            const double m = map_deriv(G, a, G.bmin[3*lb + a] + (c + 0.5)*G.dx[3*lb + a]);
            sMc[a][c + 1] = m;
            if (yonly && a == 1)
            {
                const double jc = jac_at(1.0, m, 1.0);
                sY[0][c + 1] = jc; sY[1][c + 1] = nrm_at(1.0, jc); sY[2][c + 1] = nrm_at(m, jc);
                sY[4][c + 1] = 1.0/m;
            }
        }
        else if (tid < 105)
        {
            const int a = (tid - 54)/17, c = (tid - 54) % 17;
            const double m = map_deriv(G, a, G.bmin[3*lb + a] + ((c + 0.5) - 0.5)*G.dx[3*lb + a]);
            sMf[a][c] = m;
            if (yonly && a == 1) { sY[3][c] = nrm_at(m, jac_at(1.0, m, 1.0)); sY[5][c] = 1.0/m; }
        }
    }
    const int nz = G.nc[2];
    const long long sv = G.sv;
    const int N1 = G.N[1];
    // plane (k) strides of a core column and of an x-halo column
    const long long plane = (long long)G.nc[0]*N1, xplane = (long long)N1;

    // halo cell of this thread: waves 0 and 1 own the 64 edge cells and the
    // 4 corners of the 18x18 plane (waves 2 and 3 evaluate the block-boundary faces)
    int hi = 0, hj = 0;
    const bool has_halo = tid < 68;
    if (tid < 16)      { hi = -1;       hj = tid; }
    else if (tid < 32) { hi = 16;       hj = tid - 16; }
    else if (tid < 48) { hi = tid - 32; hj = -1; }
    else if (tid < 64) { hi = tid - 48; hj = 16; }
    else if (tid < 68) { const int c = tid - 64; hi = (c & 1) ? 16 : -1; hj = (c & 2) ? 16 : -1; }
    const int pown = lpos(i, j), phalo = lpos(hi, hj);
    // left and right cell of the block-boundary face of a lane of wave 2 (x,
    // row tid - 128) or 3 (y, column tid - 192); the other lanes' own cell
    const int pbl = (tid >= 128 && tid < 144) ? lpos(15, tid - 128) : (tid >= 192 && tid < 208) ? lpos(tid - 192, 15) : pown;
    const int pbr = (tid >= 128 && tid < 144) ? lpos(16, tid - 128) : (tid >= 192 && tid < 208) ? lpos(tid - 192, 16) : pown;

    // column bases at plane k = 0; plane k is base + k*stride (the own column
    // and the residual are core columns, a halo column with hi = -1 or 16 is
    // an x-halo column)
    const long long blk = (long long)lb*G.sb;
    const double* __restrict__ Bown = prims + blk + stored_offset(G, i, j, 0);
    const double* __restrict__ Bhalo = prims + blk + stored_offset(G, hi, hj, 0);
    const long long hplane = (hi >= 0 && hi < 16) ? plane : xplane;
    // STG == 2: the halo is read from the neighbour blocks' interiors (d_nbr:
    // the block that feeds each ghost region), never from this block's ghost
    // cells; the halo column is then a core column of its x/y neighbour, and
    // planes -1 and nz come from the z neighbours (the same values an
    // exchange would have copied into the ghosts)
    const int hex = hi < 0 ? -1 : (hi > 15 ? 1 : 0), hey = hj < 0 ? -1 : (hj > 15 ? 1 : 0);
    const int* __restrict__ nbl = STG == 2 ? A.nbr + 27*lb : nullptr;
    // a y-halo cell across an isothermal wall (no source block in y): what
    // the wall fill writes there, i.e. the cell of the mirrored row (0 for the
    // low wall, nc1 - 1 for the high one) in the same column and plane,
    // itself found through the source table without the y step, with
    // T -> 2 T_wall - T and the velocity negated (boundary_fill.h)
    // (built into the mapped variant only, where the walled channel runs)
    const bool hwall = STG == 2 && MAP && has_halo && A.wall_y && hey != 0 && nbl[(hex + 1) + 3*(hey + 1) + 9] < 0;
    const int hey_s = hwall ? 0 : hey;
    const int hj_s = hwall ? (hey < 0 ? -1 - hj : 2*G.nc[1] - (hj + 1)) : hj - 16*hey;
    // (a mirrored cell of the block's own columns lies in the block itself:
    // the source table has no entry for the block's own region)
    const int src_n = (STG == 2 && has_halo)
        ? ((hex == 0 && hey_s == 0) ? lb : nbl[(hex + 1) + 3*(hey_s + 1) + 9]) : 0;
    const double* __restrict__ Bhalo_n = (STG == 2 && has_halo)
        ? prims + (long long)src_n*G.sb + stored_offset(G, hi - 16*hex, hj_s, 0)
        : Bhalo;
    auto load_ptr = [&](const double* e) -> Raw { return Raw{e[0], e[sv], e[2*sv], e[3*sv], e[4*sv]}; };
    auto load_own = [&](int ck) -> Raw
    {
        if (STG != 2 || (ck >= 0 && ck < nz)) return load_ptr(Bown + ck*plane);
        const int ez = ck < 0 ? -1 : 1;
        const long long S = nbl[1 + 3 + 9*(ez + 1)];
        return load_ptr(prims + S*G.sb + stored_offset(G, i, j, ck - ez*nz));
    };
    auto load_halo = [&](int ck) -> Raw
    {
        if (STG != 2) return load_ptr(Bhalo + ck*hplane);
        Raw r;
        if (ck >= 0 && ck < nz) r = load_ptr(Bhalo_n + ck*plane);
        else
        {
            const int ez = ck < 0 ? -1 : 1;
            const long long S = nbl[(hex + 1) + 3*(hey_s + 1) + 9*(ez + 1)];
            r = load_ptr(prims + S*G.sb + stored_offset(G, hi - 16*hex, hj_s, ck - ez*nz));
        }
        if (MAP && hwall) r = Raw{r.p, 2.0*A.t_wall - r.T, -r.u, -r.v, -r.w};
        return r;
    };
    const long long own_off = blk + stored_offset(G, i, j, 0);   // core column (i, j) at k = 0
    double* __restrict__ Rown = rhs + own_off;

    auto cell = [&](const Raw& r) -> CellV { return make_cell(C, r.p, r.T, r.u, r.v, r.w); };
    // LDS window: ring slots of velocities (rotated by pointer), scalar buffers by parity
    double* ring[3] = {sU[0], sU[1], sU[2]};      // planes k-1, k, k+1
    auto put_vel = [&](double* s, int p, const CellV& c) { s[p] = c.u; s[HP + p] = c.v; s[2*HP + p] = c.w; };
    auto put_sca = [&](double* t, int p, const CellV& c)
    {
        t[p] = c.p; t[HP + p] = c.T; t[2*HP + p] = c.rho; t[3*HP + p] = c.e;
    };

    // increment mode: the residual of the next plane to be written is requested
    // before that iteration's primitive prefetch, so waiting for it never waits
    // for the prefetch
    double rin[5];
    #pragma unroll
    for (int n = 0; n < 5; ++n) rin[n] = INC ? Rown[k0*plane + n*sv] : 0.0;

    // prologue: planes k0-1, k0, k0+1 resident; plane k0+2 in flight (one
    // plane ahead is a whole plane's arithmetic, 4 us, ahead of its use; a
    // second one only took 20 registers the fused stages spilled for)
    const CellV prev = cell(load_own(k0 - 1));
    const CellV cur0 = cell(load_own(k0));
    const CellV nxt0 = cell(load_own(k0 + 1));
    Raw nr{}, hr{};
    if (k0 + 2 <= k1) nr = load_own(k0 + 2);
    put_vel(ring[0], pown, prev);
    put_vel(ring[1], pown, cur0); put_sca(sS[0], pown, cur0);
    put_vel(ring[2], pown, nxt0); put_sca(sS[1], pown, nxt0);
    if (has_halo)
    {
        put_vel(ring[0], phalo, cell(load_halo(k0 - 1)));
        const CellV h0 = cell(load_halo(k0)), h1 = cell(load_halo(k0 + 1));
        put_vel(ring[1], phalo, h0); put_sca(sS[0], phalo, h0);
        put_vel(ring[2], phalo, h1); put_sca(sS[1], phalo, h1);
        if (k0 + 2 <= k1) hr = load_halo(k0 + 2);
    }
    lds_barrier();

    // mapped coordinates: this column's d x / d xi along x and y (cell centres)
    const double m0i = MAP ? sMc[0][i + 1] : 1.0, m1j = MAP ? sMc[1][j + 1] : 1.0;
    double zlo[5];
    constexpr bool power = S::vs && S::law == SPD_LAW_POWER;
    {
        double g[3][3], gT, mt[3] = {1.0, 1.0, 1.0};
        grads_z<S>(ring[0], ring[1], pown, prev, cur0, ix, iy, iz, g, gT);
        if constexpr (MAP)
        {
            // face k0 - 1/2: L = plane k0 - 1, R = plane k0
            const double mL = sMc[2][k0], mR = sMc[2][k0 + 1], mf = sMf[2][k0];
            if constexpr (yonly) { mt[0] = mt[1] = mt[2] = sY[1][j + 1]; }
            else
            {
                mt[0] = nrm_at(mL, jac_at(m0i, m1j, mL));
                mt[1] = nrm_at(mR, jac_at(m0i, m1j, mR));
                mt[2] = nrm_at(mf, jac_at(m0i, m1j, mf));
            }
            if constexpr (yonly) grads_map_y<2>(g, gT, m1j, sY[4][j + 1]);
            else grads_map<2>(G, g, gT, mf, m0i, m1j);
        }
        double pw[1] = {1.0};
        if constexpr (power)
        {
            const double x[1] = {pow_arg(C, prev.T + cur0.T)};
            pow_faces<1>(C.ps, x, C.power, false, pw);
        }
        face_product<2, S, (MAP != 0)>(C, prev, cur0, g, gT, iz, mt, zlo, pw[0]);
    }

    // One plane k: every face, the residual of its cells, and the entry of
    // plane k+2 (from nr / hr, which are then refilled with plane k+3).
    auto plane_step = [&](int k)
    {
        // the x pushes staged by plane k-1 (visible since its last barrier;
        // the staging buffer is refilled only after this plane's first barrier)
        if (STG && A.push_ghosts && k > k0) flush_x(G, A.push, A.qout, xs, lb, k - 1);
        const double* sm = ring[0];
        const double* s0 = ring[1];
        const double* sp = ring[2];
        const double* sk = sS[(k - k0) & 1];
        // the cells of this column in planes k and k+1, from the window
        const CellV cur = cell_from_lds(sk, s0, pown);
        const CellV nxt = cell_from_lds(sS[(k - k0 + 1) & 1], sp, pown);
        // the power law of the thread's three faces and, in waves 2 and 3, of
        // its block-boundary face
        double pw[4] = {1.0, 1.0, 1.0, 1.0};
        if constexpr (power)
        {
            const double* sT = sk + HP;
            double x[4] = {pow_arg(C, sT[pown - 1] + cur.T), pow_arg(C, sT[pown - HX] + cur.T),
                           pow_arg(C, cur.T + nxt.T), 1.0};
            const bool closing = __builtin_amdgcn_readfirstlane(tid) >= 128;
            if (closing) x[3] = pow_arg(C, sT[pbl] + sT[pbr]);
            pow_faces<3>(C.ps, x, C.power, closing, pw);
        }
        double zhi[5];
        // this cell's own low x- and y-face products (the LDS copies serve
        // the neighbour cells that share those faces); the residual reads
        // them from registers where that fits the register budget (plain
        // flux_div on identity coordinates without pressure dissipation)
        double px[5], py[5];
        constexpr bool own_reg = STG == 0 && !MAP && !S::pd;
        // mapped coordinates: plane k's d z / d zeta and this cell's Jacobian
        const double m2k = MAP ? sMc[2][k + 1] : 1.0;
        const double jc = MAP ? (yonly ? sY[0][j + 1] : jac_at(m0i, m1j, m2k)) : 1.0;
        // the three faces of all lanes, then the block-boundary x-faces
        // (wave 2) and y-faces (wave 3); the series pow has no branch, so the
        // three faces form one straight-line block
        {
            // low x-face of (i,j): L = (i-1, j)
            const int pL = pown - 1;
            const CellV L = cell_from_lds(sk, s0, pL);
            double g[3][3], gT, mt[3] = {1.0, 1.0, 1.0};
            grads_x<S>(sm, s0, sp, pL, pown, L, cur, ix, iy, iz, g, gT);
            if constexpr (MAP)
            {
                const double mL = sMc[0][i], mf = sMf[0][i];
                if constexpr (yonly) { mt[0] = mt[1] = mt[2] = sY[1][j + 1]; }
                else
                {
                    mt[0] = nrm_at(mL, jac_at(mL, m1j, m2k));
                    mt[1] = nrm_at(m0i, jc);
                    mt[2] = nrm_at(mf, jac_at(mf, m1j, m2k));
                }
                if constexpr (yonly) grads_map_y<0>(g, gT, m1j, sY[4][j + 1]);
                else grads_map<0>(G, g, gT, mf, m1j, m2k);
            }
            face_product<0, S, (MAP != 0)>(C, L, cur, g, gT, ix, mt, px, pw[0]);
            for (int n = 0; n < 5; ++n) sFx[n][j*17 + i] = px[n];
        }
        {
            // low y-face of (i,j): L = (i, j-1)
            const int pL = pown - HX;
            const CellV L = cell_from_lds(sk, s0, pL);
            double g[3][3], gT, mt[3] = {1.0, 1.0, 1.0};
            grads_y<S>(sm, s0, sp, pL, pown, L, cur, ix, iy, iz, g, gT);
            if constexpr (MAP)
            {
                const double mL = sMc[1][j], mf = sMf[1][j];
                if constexpr (yonly) { mt[0] = sY[2][j]; mt[1] = sY[2][j + 1]; mt[2] = sY[3][j]; }
                else
                {
                    mt[0] = nrm_at(mL, jac_at(m0i, mL, m2k));
                    mt[1] = nrm_at(m1j, jc);
                    mt[2] = nrm_at(mf, jac_at(m0i, mf, m2k));
                }
                if constexpr (yonly) grads_map_y<1>(g, gT, mf, sY[5][j]);
                else grads_map<1>(G, g, gT, mf, m2k, m0i);
            }
            face_product<1, S, (MAP != 0)>(C, L, cur, g, gT, iy, mt, py, pw[1]);
            for (int n = 0; n < 5; ++n) sFy[n][j*16 + i] = py[n];
        }
        {
            // high z-face k+1/2: L = (i,j,k), R = (i,j,k+1)
            double g[3][3], gT, mt[3] = {1.0, 1.0, 1.0};
            grads_z<S>(s0, sp, pown, cur, nxt, ix, iy, iz, g, gT);
            if constexpr (MAP)
            {
                const double mR = sMc[2][k + 2], mf = sMf[2][k + 1];
                if constexpr (yonly) { mt[0] = mt[1] = mt[2] = sY[1][j + 1]; }
                else
                {
                    mt[0] = nrm_at(m2k, jc);
                    mt[1] = nrm_at(mR, jac_at(m0i, m1j, mR));
                    mt[2] = nrm_at(mf, jac_at(m0i, m1j, mf));
                }
                if constexpr (yonly) grads_map_y<2>(g, gT, m1j, sY[4][j + 1]);
                else grads_map<2>(G, g, gT, mf, m0i, m1j);
            }
            face_product<2, S, (MAP != 0)>(C, cur, nxt, g, gT, iz, mt, zhi, pw[2]);
        }
        if (tid >= 128 && tid < 144)
        {
            // block-boundary x-faces (16 - 1/2, jj)
            const int jj = tid - 128;
            const int pL = lpos(15, jj), pR = lpos(16, jj);
            const CellV L = cell_from_lds(sk, s0, pL), Rr = cell_from_lds(sk, s0, pR);
            double g[3][3], gT, P[5], mt[3] = {1.0, 1.0, 1.0};
            grads_x<S>(sm, s0, sp, pL, pR, L, Rr, ix, iy, iz, g, gT);
            if constexpr (MAP)
            {
                const double m1 = sMc[1][jj + 1], mL = sMc[0][16], mR = sMc[0][17], mf = sMf[0][16];
                if constexpr (yonly) { mt[0] = mt[1] = mt[2] = sY[1][jj + 1]; }
                else
                {
                    mt[0] = nrm_at(mL, jac_at(mL, m1, m2k));
                    mt[1] = nrm_at(mR, jac_at(mR, m1, m2k));
                    mt[2] = nrm_at(mf, jac_at(mf, m1, m2k));
                }
                if constexpr (yonly) grads_map_y<0>(g, gT, m1, sY[4][jj + 1]);
                else grads_map<0>(G, g, gT, mf, m1, m2k);
            }
            face_product<0, S, (MAP != 0)>(C, L, Rr, g, gT, ix, mt, P, pw[3]);
            for (int n = 0; n < 5; ++n) sFx[n][jj*17 + 16] = P[n];
        }
        if (tid >= 192 && tid < 208)
        {
            // block-boundary y-faces (ii, 16 - 1/2)
            const int ii = tid - 192;
            const int pL = lpos(ii, 15), pR = lpos(ii, 16);
            const CellV L = cell_from_lds(sk, s0, pL), Rr = cell_from_lds(sk, s0, pR);
            double g[3][3], gT, P[5], mt[3] = {1.0, 1.0, 1.0};
            grads_y<S>(sm, s0, sp, pL, pR, L, Rr, ix, iy, iz, g, gT);
            if constexpr (MAP)
            {
                const double m0 = sMc[0][ii + 1], mL = sMc[1][16], mR = sMc[1][17], mf = sMf[1][16];
                if constexpr (yonly) { mt[0] = sY[2][16]; mt[1] = sY[2][17]; mt[2] = sY[3][16]; }
                else
                {
                    mt[0] = nrm_at(mL, jac_at(m0, mL, m2k));
                    mt[1] = nrm_at(mR, jac_at(m0, mR, m2k));
                    mt[2] = nrm_at(mf, jac_at(m0, mf, m2k));
                }
                if constexpr (yonly) grads_map_y<1>(g, gT, mf, sY[5][16]);
                else grads_map<1>(G, g, gT, mf, m2k, m0);
            }
            face_product<1, S, (MAP != 0)>(C, L, Rr, g, gT, iy, mt, P, pw[3]);
            for (int n = 0; n < 5; ++n) sFy[n][16*16 + ii] = P[n];
        }
        #pragma unroll
        for (int n = 0; n < 5; ++n) keep_here(zhi[n]);
        // a fused stage's earlier residuals of cell (i,j,k), requested before
        // the barrier so that their latency overlaps the wait for the other waves
        double rprev[2][5];
        if constexpr (STG)
        {
            const long long co = own_off + k*plane;
            #pragma unroll
            for (int t = 0; t < 2; ++t)
            {
                if (t + 1 >= A.n || A.c[t] == 0.0) continue;
                #pragma unroll
                for (int v = 0; v < 5; ++v) rprev[t][v] = A.r[t][co + v*sv];
            }
        }
        lds_barrier();

        // rhs of cell (i,j,k): faces in the order x-, x+, y-, y+, z-, z+
        // (flux_div_basic.h:54-72; the high faces enter as -P)
        double* __restrict__ ro = Rown + k*plane;
        // identity coordinates: the face products already carry 1/dx; mapped:
        // each cell scales the (composition-scaled) face fluxes by its own
        // jac/dx, i.e. s = jac (1 - 2 pm) inv_dx (flux_div_basic.h:66-68)
        double fx = 1.0, fy = 1.0, fz = 1.0;
        if constexpr (MAP)
        {
            const double sc = S::keep ? 0.125 : 1.0;
            fx = sc*(jc*ix); fy = sc*(jc*iy); fz = sc*(jc*iz);
        }
        double rr[5];
        #pragma unroll
        for (int n = 0; n < 5; ++n)
        {
            double r = rin[n];
            if constexpr (MAP)
            {
                r += sFx[n][j*17 + i]*fx;
                r -= sFx[n][j*17 + i + 1]*fx;
                r += sFy[n][j*16 + i]*fy;
                r -= sFy[n][(j + 1)*16 + i]*fy;
                r += zlo[n]*fz;
                r -= zhi[n]*fz;
            }
            else
            {
                r += own_reg ? px[n] : sFx[n][j*17 + i];
                r -= sFx[n][j*17 + i + 1];
                r += own_reg ? py[n] : sFy[n][j*16 + i];
                r -= sFy[n][(j + 1)*16 + i];
                r += zlo[n];
                r -= zhi[n];
            }
            // streamed: nothing in this launch reads it again
            if (!STG || A.store_rhs) __builtin_nontemporal_store(r, ro + n*sv);
            rr[n] = r;
            zlo[n] = zhi[n];
        }
        if constexpr (STG)
        {
            // the stage of cell (i,j,k): its stored primitives are the window's
            const long long co = own_off + k*plane;
            // p2c and c2p of spd_stage.hpp, their quotients without the ends of
            // the range; the cell's density is the window's where the stage
            // converts with the flux's gas constant
            double rho = cur.rho;
            if (!A.same_R) rho = quot_inf(cur.p, A.R*cur.T);
            const double rhoU2 = rho*(cur.u*cur.u + cur.v*cur.v + cur.w*cur.w);
            const double gm1 = A.gamma - 1.0;
            double qq[5], cons[5] = {rho, 0.5*rhoU2 + __builtin_amdgcn_div_fixup(div_const(cur.p, gm1, A.inv_gm1), gm1, cur.p),
                                     rho*cur.u, rho*cur.v, rho*cur.w};
            #pragma unroll
            for (int t = 0; t < 2; ++t)
            {
                if (t + 1 >= A.n || A.c[t] == 0.0) continue;
                double inc[5];
                #pragma unroll
                for (int v = 0; v < 5; ++v) inc[v] = A.c[t]*rprev[t][v];
                #pragma unroll
                for (int v = 0; v < 5; ++v) cons[v] += inc[v];
            }
            const double cl = A.c[A.n - 1];
            if (cl != 0.0)
            {
                double inc[5];
                #pragma unroll
                for (int v = 0; v < 5; ++v) inc[v] = cl*rr[v];
                #pragma unroll
                for (int v = 0; v < 5; ++v) cons[v] += inc[v];
            }
            {
                const double invrho = quot_inf(1.0, cons[0]);
                qq[2] = invrho*cons[2]; qq[3] = invrho*cons[3]; qq[4] = invrho*cons[4];
                const double ru2 = cons[0]*(qq[2]*qq[2] + qq[3]*qq[3] + qq[4]*qq[4]);
                qq[0] = gm1*(cons[1] - 0.5*ru2);
                qq[1] = quot_inf(qq[0], A.R*cons[0]);
            }
            #pragma unroll
            for (int v = 0; v < 5; ++v) __builtin_nontemporal_store(qq[v], A.qout + co + v*sv);
            if (A.push_ghosts)
            {
                const CellIt c{i, j, k, lb};
                push_ghosts(G, A.push, A.qout, c, qq, true);
                stage_x(G, xs, c, qq);
            }
        }

        if (k + 1 < k1)
        {
            // plane k+2 (<= k1) enters into the ring slot of plane k-1 and the
            // parity buffer of plane k; its raw registers take plane k+3
            double* s_new = ring[0];
            ring[0] = ring[1]; ring[1] = ring[2]; ring[2] = s_new;
            double* t_new = sS[(k - k0) & 1];
            if (INC)
            {
                #pragma unroll
                for (int n = 0; n < 5; ++n) rin[n] = ro[plane + n*sv];
            }
            const CellV c2 = cell(nr);
            put_vel(s_new, pown, c2); put_sca(t_new, pown, c2);
            if (k + 3 <= k1) nr = load_own(k + 3);
            if (has_halo)
            {
                const CellV h = cell(hr);
                put_vel(s_new, phalo, h); put_sca(t_new, phalo, h);
                if (k + 3 <= k1) hr = load_halo(k + 3);
            }
        }
        lds_barrier();
    };

    for (int k = k0; k < k1; ++k) plane_step(k);
    if (STG && A.push_ghosts) flush_x(G, A.push, A.qout, xs, lb, k1 - 1);   // after the last plane's closing barrier
}

// Workgroups per block, each marching over its share of the block's planes:
// the least of rounds x (planes of a share + 0.65), with rounds the
// workgroups over those resident at once (two per CU) and 0.65 planes the cost
// of a share's prologue (256^3: 495, 514 and 550 us in 1, 2 and 4 shares).  64
// blocks take 8 shares (one round of 512 workgroups; 64^3 ten steps 557 us, 669 in
// 4 shares, 1076 in 2, 1935 whole), 576 blocks 4, 4096 blocks stay whole.
// SPD_FAST_ZSPLIT=n forces the choice.
int fast_zsplit(const Grid& g)
{
    const int nz = g.geom.nc[2], most = std::min(nz, 255);
    if (const char* e = getenv("SPD_FAST_ZSPLIT")) return std::max(1, std::min(most, atoi(e)));
    const long slots = 2L*g.ctx->cus, nb = g.geom.nblk;
    int best = 1;
    double best_cost = 1e300;
    for (int zs = 1; zs <= most; ++zs)
    {
        const double cost = (double)((zs*nb + slots - 1)/slots)*((nz + zs - 1)/zs + 0.65);
        if (cost < best_cost - 1e-9) { best_cost = cost; best = zs; }
    }
    return best;
}

// Workgroup order of a launch: contiguous runs of blocks per XCD (1) or the
// launch order (0).  Runs pay where other workgroups read the same lines:
// a block that reads its halo from the neighbour blocks' interiors (fused
// stages on periodic identity grids: on the 256^3 Taylor-Green step they
// halve the lines those stages fetch into L2, 2.97 -> 1.54 GB per launch, and
// save 2% of the step), or a block split between workgroups, whose parts
// re-read the planes next to their shares (the 192x128x96 channel flux_div,
// 4 parts per block: 1-3.5% faster in alternating runs on one GPU).  A whole block that reads its own ghost
// cells shares nothing with its neighbours, and flux_div times the same
// either way.  SPD_FAST_XCD=0|1 forces the choice.
int fast_xcd_runs(bool shared_reads)
{
    if (const char* e = getenv("SPD_FAST_XCD")) return e[0] == '1' ? 1 : 0;
    return shared_reads ? 1 : 0;
}

template <int KEEP, int PDISS, int VISC>
void launch_fast(const Grid& g, const double* prims, double* rhs, const FastCfg& C, bool increment, hipStream_t s)
{
    const int zs = fast_zsplit(g);
    const int xr = fast_xcd_runs(zs > 1) ? 0x100 : 0;
    auto go = [&](auto kernel)
    {
        hipLaunchKernelGGL(kernel, dim3(g.geom.nblk*zs), dim3(256), 0, s, g.geom, prims, rhs, C, StageArgs{}, zs | xr);
    };
    switch (map_variant(g.geom) + (increment ? 3 : 0))
    {
        case 0: go(k_flux_fast<KEEP, PDISS, VISC, false, 0>); break;
        case 1: go(k_flux_fast<KEEP, PDISS, VISC, false, 1>); break;
        case 2: go(k_flux_fast<KEEP, PDISS, VISC, false, 2>); break;
        case 3: go(k_flux_fast<KEEP, PDISS, VISC, true, 0>); break;
        case 4: go(k_flux_fast<KEEP, PDISS, VISC, true, 1>); break;
        case 5: go(k_flux_fast<KEEP, PDISS, VISC, true, 2>); break;
    }
    SPD_LAUNCH_CHECK();
}

template <int KEEP, int PDISS>
bool dispatch_visc(int visc, const Grid& g, const double* prims, double* rhs, const FastCfg& C, bool inc, hipStream_t s)
{
    switch (visc)
    {
        case 0: if (KEEP || PDISS) { launch_fast<KEEP, PDISS, 0>(g, prims, rhs, C, inc, s); return true; } return false;
        case 1: launch_fast<KEEP, PDISS, 1>(g, prims, rhs, C, inc, s); return true;
        case 2: launch_fast<KEEP, PDISS, 2>(g, prims, rhs, C, inc, s); return true;
    }
    return false;
}

template <int KEEP, int PDISS, int VISC>
void launch_fast_stage(const Grid& g, const double* qin, double* rhs, const FastCfg& C, const StageArgs& A,
                       bool read_neighbours, hipStream_t s)
{
    const int zs = fast_zsplit(g);
    const int xr = fast_xcd_runs(read_neighbours || zs > 1) ? 0x100 : 0;
    auto go = [&](auto kernel)
    {
        hipLaunchKernelGGL(kernel, dim3(g.geom.nblk*zs), dim3(256), 0, s, g.geom, qin, rhs, C, A, zs | xr);
    };
    switch (map_variant(g.geom) + (read_neighbours ? 3 : 0))
    {
        case 0: go(k_flux_fast<KEEP, PDISS, VISC, false, 0, 1>); break;
        case 1: go(k_flux_fast<KEEP, PDISS, VISC, false, 1, 1>); break;
        case 2: go(k_flux_fast<KEEP, PDISS, VISC, false, 2, 1>); break;
        case 3: go(k_flux_fast<KEEP, PDISS, VISC, false, 0, 2>); break;
        case 4: go(k_flux_fast<KEEP, PDISS, VISC, false, 1, 2>); break;
        case 5: go(k_flux_fast<KEEP, PDISS, VISC, false, 2, 2>); break;
    }
    SPD_LAUNCH_CHECK();
}

template <int KEEP, int PDISS>
bool dispatch_visc_stage(int visc, const Grid& g, const double* qin, double* rhs, const FastCfg& C,
                         const StageArgs& A, bool nb, hipStream_t s)
{
    switch (visc)
    {
        case 0: if (KEEP || PDISS) { launch_fast_stage<KEEP, PDISS, 0>(g, qin, rhs, C, A, nb, s); return true; } return false;
        case 1: launch_fast_stage<KEEP, PDISS, 1>(g, qin, rhs, C, A, nb, s); return true;
        case 2: launch_fast_stage<KEEP, PDISS, 2>(g, qin, rhs, C, A, nb, s); return true;
    }
    return false;
}

} // namespace

namespace {

// Selects the fast kernel for (grid, flux); false when the tiled or the generic kernel runs.
bool select_fast(const DevGeom& G, const spd_flux_desc& f, int& keep, int& pd, int& vs, FastCfg& C)
{
    // identity or diagonal (tanh) maps; a 16 x 16 cross-section
    if (G.nc[0] != 16 || G.nc[1] != 16 || G.ng < 1) return false;
    for (int a = 0; a < 3; ++a) if (G.map_kind[a] != SPD_MAP_IDENTITY && G.map_kind[a] != SPD_MAP_TANH) return false;
    // the metric tables hold 16 planes; they are not read where only y is mapped
    if (map_variant(G) == 2 && G.nc[2] > 16) return false;
    if (const char* e = getenv("SPD_DISABLE_FAST")) if (e[0] == '1') return false;
    // terms must be a subsequence of [keep2, pdiss, visc] in that order
    keep = 0; pd = 0; vs = 0;
    int stage = 0;
    C = FastCfg{};
    cfg_gas(C, f);
    bool has_keep = false;
    for (int m = 0; m < f.nterms; ++m) has_keep |= f.terms[m].kind == SPD_TERM_KEEP;
    const double sc = has_keep ? 8.0 : 1.0;   // composition scale (see face_product)
    for (int m = 0; m < f.nterms; ++m)
    {
        const spd_flux_term& t = f.terms[m];
        if (t.kind == SPD_TERM_KEEP && t.order == 2 && stage < 1) { keep = 1; stage = 1; }
        else if (t.kind == SPD_TERM_PDISS && stage < 2)
        {
            pd = 1 + t.sensor; stage = 2;
            cfg_pdiss(C, t, sc);
        }
        else if (t.kind == SPD_TERM_VISC && stage < 3)
        {
            if (t.sgs != SPD_SGS_NONE) return false;   // the tiled kernel evaluates subgrid models
            vs = 1 + t.law; stage = 3;
            cfg_visc(C, t, sc);
            if (t.law == SPD_LAW_POWER && !(t.T_ref > 0.0 && t.prandtl > 0.0)) return false;
        }
        else return false;
    }
    return true;
}

} // namespace

bool flux_div_fast_eligible(const Grid& g, const spd_flux_desc& f)
{
    int keep, pd, vs;
    FastCfg C;
    return select_fast(g.geom, f, keep, pd, vs, C);
}

bool launch_flux_div_fast(const Grid& g, const double* prims, double* rhs, const spd_flux_desc& f,
                          bool increment, hipStream_t s)
{
    int keep, pd, vs;
    FastCfg C;
    if (!select_fast(g.geom, f, keep, pd, vs, C)) return false;
    bool ok = false;
    switch (keep*3 + pd)
    {
        case 0: ok = dispatch_visc<0, 0>(vs, g, prims, rhs, C, increment, s); break;
        case 1: ok = dispatch_visc<0, 1>(vs, g, prims, rhs, C, increment, s); break;
        case 2: ok = dispatch_visc<0, 2>(vs, g, prims, rhs, C, increment, s); break;
        case 3: ok = dispatch_visc<1, 0>(vs, g, prims, rhs, C, increment, s); break;
        case 4: ok = dispatch_visc<1, 1>(vs, g, prims, rhs, C, increment, s); break;
        case 5: ok = dispatch_visc<1, 2>(vs, g, prims, rhs, C, increment, s); break;
    }
    return ok;
}

// The fused stage needs the x-staged push (16 x 16 cross-sections, ng <= 2,
// nz >= 2 ng) beside the fast kernel's own conditions
static bool stage_geometry(const DevGeom& G)
{
    return G.nc[0] == 16 && G.nc[1] == 16 && G.ng >= 1 && G.ng <= 2 && G.nc[2] >= 2*G.ng;
}

// A stage can read its halo from the neighbour blocks' interiors when every
// ghost region has a source block (each axis periodic) or, on diagonal
// (mapped) coordinates, along y only is an isothermal wall the caller fills on
// both faces (wall_mask bits 2 and 3), whose ghosts the kernel forms from the
// mirrored cells (the walled channel; the identity-coordinate kernel is built
// without the wall step)
bool stage_reads_neighbours_ok(const Grid& g, int wall_mask)
{
    const bool xz = g.desc.periodic[0] && g.desc.periodic[2];
    if (g.geom.identity) return xz && g.desc.periodic[1];
    return xz && (g.desc.periodic[1] || ((wall_mask >> 2) & 3) == 3);
}

bool flux_stage_fast_eligible(const Grid& g, const spd_flux_desc& f)
{
    int keep, pd, vs;
    FastCfg C;
    if (!stage_geometry(g.geom) || !select_fast(g.geom, f, keep, pd, vs, C)) return false;
    return keep || pd || vs;
}

bool launch_flux_stage_fast(const Grid& g, const double* qin, double* qout, double* rhs, const spd_flux_desc& f,
                            const double* const* rprev, const double* coef, int nr, bool store_rhs,
                            double gamma, double R, hipStream_t s, bool read_neighbours, bool push,
                            int wall_mask, double t_wall)
{
    int keep, pd, vs;
    FastCfg C;
    if (!stage_geometry(g.geom) || !select_fast(g.geom, f, keep, pd, vs, C)) return false;
    if (nr < 1 || nr > 3) throw ArgError{"a fused stage combines 1..3 residuals"};
    if (qin == qout) throw ArgError{"a fused stage needs distinct input and output arrays"};
    if (read_neighbours && !stage_reads_neighbours_ok(g, wall_mask))
        throw ArgError{"neighbour-read stages need every axis periodic, or on mapped coordinates y walled on both faces"};
    StageArgs A{};
    A.qout = qout;
    for (int t = 0; t + 1 < nr; ++t) A.r[t] = rprev[t];
    for (int t = 0; t < nr; ++t) A.c[t] = coef[t];
    A.n = nr;
    A.store_rhs = store_rhs ? 1 : 0;
    A.gamma = gamma; A.R = R; A.inv_gm1 = 1.0/(gamma - 1.0);
    A.same_R = R == C.R ? 1 : 0;
    A.push = g.d_push;
    A.push_ghosts = push ? 1 : 0;
    A.nbr = g.d_nbr;
    A.wall_y = (read_neighbours && !g.desc.periodic[1]) ? 1 : 0;
    A.t_wall = t_wall;
    bool ok = false;
    switch (keep*3 + pd)
    {
        case 0: ok = dispatch_visc_stage<0, 0>(vs, g, qin, rhs, C, A, read_neighbours, s); break;
        case 1: ok = dispatch_visc_stage<0, 1>(vs, g, qin, rhs, C, A, read_neighbours, s); break;
        case 2: ok = dispatch_visc_stage<0, 2>(vs, g, qin, rhs, C, A, read_neighbours, s); break;
        case 3: ok = dispatch_visc_stage<1, 0>(vs, g, qin, rhs, C, A, read_neighbours, s); break;
        case 4: ok = dispatch_visc_stage<1, 1>(vs, g, qin, rhs, C, A, read_neighbours, s); break;
        case 5: ok = dispatch_visc_stage<1, 2>(vs, g, qin, rhs, C, A, read_neighbours, s); break;
    }
    return ok;
}

} // namespace spd
