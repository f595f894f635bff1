// mfc_viscous.hip -- the RHS and RK stage of viscous runs: inviscid and
// viscous fluxes, with velocity gradients by finite differences or
// (weno_Re_flux) by the divergence theorem on WENO face values.
//
// The viscous flux needs, per face, the HLLC star velocity and the
// reconstructed volume fractions (m_riemann_solvers.fpp:169-231, :313-323),
// which the inviscid sweeps keep in registers and LDS only.  Viscous runs
// therefore use these kernels in place of the sweeps.  The face kernels
// reconstruct with the sweeps' own weno_cell and hllc_face (hence the same
// bits), each cell converted to primitive once into an LDS tile and
// reconstructed once (both faces), one variable at a time.  The
// finite-difference gradients come from the primitive velocities (of the
// tile, and for the x faces' neighbours in y of the conservative field);
// with weno_Re_flux, gradient planes computed by a pass before the
// directions are reconstructed in the tile too.  Per face they form the HLLC
// flux, the contact velocity and the viscous source flux
// (m_riemann_solvers.fpp:683-902), and then finish the cells between their
// faces: the flux divergence, the alpha*div(u) source and the viscous
// divergence in the reference's order (m_rhs.fpp:565-652), and in the last
// direction the RK stage.
#include "mfc_viscous.hpp"

namespace mfc {

namespace {

__device__ __forceinline__ long goff(const ViscArgs &a, int i, int j) {
    return (long)(i + a.b) + a.nxg * (long)(j + a.bj);
}

// Velocity component d of cell (i, j) as cons->prim computes it
// (m_variables_conversion.fpp:349-357): rho = max(sum alpha_i rho_i, sgm_eps).
template <int NF, int D>
__device__ __forceinline__ double cell_vel(const ViscArgs &a, int i, int j, int d) {
    const long o = goff(a, i, j);
    double rho = 0.0;
#pragma unroll
    for (int f = 0; f < NF; ++f) rho = rho + a.q.v[f][o];
    rho = max_ref(rho, 1e-16);
    return a.q.v[Sys<NF, D>::MOM + d][o] / rho;
}

// Harmonic face Reynolds numbers (m_riemann_solvers.fpp:169-231).
template <int NF, int D>
__device__ __forceinline__ void re_avg(const ViscArgs &a, const double *ql, const double *qr, double *ra) {
    using Y = Sys<NF, D>;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        ra[r] = 0.0;
        if (a.vp.size[r] == 0) continue;
        double reL = 0.0, reR = 0.0;
        for (int q = 0; q < a.vp.size[r]; ++q) {
            reL = ql[Y::ADV + a.vp.idx[r][q]] / a.vp.res[r][q] + reL;
            reR = qr[Y::ADV + a.vp.idx[r][q]] / a.vp.res[r][q] + reR;
        }
        reL = 1.0 / max_ref(reL, 1e-16);
        reR = 1.0 / max_ref(reR, 1e-16);
        ra[r] = 2.0 / (1.0 / reL + 1.0 / reR);
    }
}

// WENO coefficients of cell c of the direction: kernel arguments (scalar
// registers) on uniform grids, as in the sweeps, else per-cell loads; the
// same values either way.
template <bool UNI>
__device__ __forceinline__ void cell_coef(const ViscArgs &a, int c, double *cf) {
#pragma unroll
    for (int q = 0; q < kNCoef; ++q) cf[q] = UNI ? a.ucf[q] : a.coef[(long)q * a.ncell + (c + a.b)];
}

// Viscous source flux of one face (m_riemann_solvers.fpp:683-902) from its
// two face states, star velocity and the face averages of the velocity
// gradients: ax[c] = dvel_avg_dx(c), ay[c] = dvel_avg_dy(c), each
// 5e-1*(solver-left + solver-right value) as the reference forms it (the
// solver's left gradients are the caller's dqR_prim_d*_n, m_rhs.fpp:545-556).
template <int NF, int D, int DIR>
__device__ __forceinline__ void face_flux(const ViscArgs &a, const double *ql, const double *qr, const double *ax,
                                          const double *ay, double *flux, double &ustar, double *fs) {
    double vsrc[D];
    hllc_face<NF, D, DIR, double, true>(ql, qr, a.eos, flux, ustar, vsrc);
    double ra[2];
    re_avg<NF, D>(a, ql, qr, ra);
#pragma unroll
    for (int v = 0; v <= D; ++v) fs[v] = 0.0;
    if constexpr (DIR == 0) {
        if (a.vp.size[0] > 0) {
            const double t11 = (4.0 / 3.0) * ax[0] / ra[0];
            fs[0] = fs[0] - t11;
            fs[D] = fs[D] - vsrc[0] * t11;
        }
        if (a.vp.size[1] > 0) {
            const double t11 = ax[0] / ra[1];
            fs[0] = fs[0] - t11;
            fs[D] = fs[D] - vsrc[0] * t11;
        }
        if constexpr (D == 2) {
            if (a.vp.size[0] > 0) {
                double tau[2];
                tau[0] = -((2.0 / 3.0) * ay[1] / ra[0]);
                tau[1] = (ay[0] + ax[1]) / ra[0];
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    fs[d] = fs[d] - tau[d];
                    fs[D] = fs[D] - vsrc[d] * tau[d];
                }
            }
            if (a.vp.size[1] > 0) {
                const double t11 = ay[1] / ra[1];
                fs[0] = fs[0] - t11;
                fs[D] = fs[D] - vsrc[0] * t11;
            }
        }
    } else {
        if (a.vp.size[0] > 0) {
            double tau[2];
            tau[0] = (ay[0] + ax[1]) / ra[0];
            tau[1] = (4.0 * ay[1] - 2.0 * ax[0]) / (3.0 * ra[0]);
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                fs[d] = fs[d] - tau[d];
                fs[D] = fs[D] - vsrc[d] * tau[d];
            }
        }
        if (a.vp.size[1] > 0) {
            const double t22 = (ax[0] + ay[1]) / ra[1];
            fs[1] = fs[1] - t22;
            fs[D] = fs[D] - vsrc[1] * t22;
        }
    }
}

// Face averages of finite-difference gradients: both sides of a face hold
// the same difference (dqR_prim_d*_n of the left cell and dqL_prim_d*_n of
// the right one, m_viscous.fpp:231-336), so each average is 5e-1*(g + g).
// gn: differences across the face, gt: the transverse four-point averages.
template <int D, int DIR>
__device__ __forceinline__ void fd_averages(const double *gn, const double *gt, double *ax, double *ay) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const double n2 = 5e-1 * (gn[c] + gn[c]), t2 = 5e-1 * (gt[c] + gt[c]);
        ax[c] = DIR == 0 ? n2 : t2;
        ay[c] = DIR == 0 ? t2 : n2;
    }
}

// Holds a variable's face states where they are computed: without it the
// compiler starts every variable's reconstruction before it ends the first.
__device__ __forceinline__ void pin(double &l, double &r) { asm volatile("" : "+v"(l), "+v"(r)); }

// Finish of one cell, in the reference's order (m_rhs.fpp:565-652): the flux
// divergence (assigned in the first direction, added after), the alpha*div(u)
// source, the viscous divergence of momentum and energy; then the rhs store,
// or the RK stage in the last direction (the sweeps' rk_combine arithmetic).
// d: lower minus upper face of the S fluxes, dus: upper minus lower contact
// velocity, dv: lower minus upper face of the viscous fluxes.
template <int NF, int D>
__device__ __forceinline__ void visc_finish(const SweepArgs &s, int i, int j, double inv, const double *d, double dus,
                                            const double *dv) {
    using Y = Sys<NF, D>;
    constexpr int S = Y::S;
    const long go = ghost_off(s, i, j, 0), t = (long)j * (s.m + 1) + i;
    double r[S];
#pragma unroll
    for (int v = 0; v < S; ++v) r[v] = s.accumulate ? s.rhs.v[v][t] + inv * d[v] : inv * d[v];
#pragma unroll
    for (int k = 0; k < NF; ++k) r[Y::ADV + k] = r[Y::ADV + k] + inv * s.qin.v[Y::ADV + k][go] * dus;
#pragma unroll
    for (int v = 0; v <= D; ++v) r[Y::MOM + v] = r[Y::MOM + v] + inv * dv[v];
    if (s.rk == kRkNone) {
#pragma unroll
        for (int v = 0; v < S; ++v) s.rhs.v[v][t] = r[v];
        return;
    }
    // combined and stored per variable (rk_combine's arithmetic; its results in
    // an array stayed in scratch memory here)
    switch (s.rk) {
    case kRkEuler:
#pragma unroll
        for (int v = 0; v < S; ++v) s.qout.v[v][go] = s.qbase.v[v][go] + s.dt * r[v];
        break;
    case kRk2Final:
#pragma unroll
        for (int v = 0; v < S; ++v) s.qout.v[v][go] = (s.qbase.v[v][go] + s.qin.v[v][go] + s.dt * r[v]) / 2.0;
        break;
    case kRk3Stage2:
#pragma unroll
        for (int v = 0; v < S; ++v) s.qout.v[v][go] = (3.0 * s.qbase.v[v][go] + s.qin.v[v][go] + s.dt * r[v]) / 4.0;
        break;
    default:
#pragma unroll
        for (int v = 0; v < S; ++v)
            s.qout.v[v][go] = third(s.qbase.v[v][go] + 2.0 * s.qin.v[v][go] + 2.0 * s.dt * r[v]);
        break;
    }
}

// The face average of gradient plane values reconstructed at the upper face of
// the left cell (R, dqR_prim_d*_n) and the lower face of the right cell (L,
// dqL_prim_d*_n), with the bc = -4 copies of
// s_populate_riemann_states_variables_buffers (m_riemann_solvers.fpp:488-608,
// with the caller's L/R swap), then 5e-1*(R + L) as
// s_compute_viscous_source_flux averages them (:683-902).
__device__ __forceinline__ double grad_average(const ViscArgs &a, int f, int s, double R, double L) {
    if (f == -1 && a.bc_beg == -4) R = L;
    if (f == s && a.bc_end == -4) L = R;
    return 5e-1 * (R + L);
}

// Gradient planes of every direction (weno_Re_flux), one thread per ghosted
// cell: each velocity component reconstructed along direction e with WENO over
// cells [-b+polyn, s+b-polyn] (s_reconstruct_cell_boundary_values_visc,
// m_viscous.fpp:400-469), then d u_c / d x_e = 1/ds * (vR - vL)
// (s_apply_scalar_divergence_theorem, :372-398) over [-b+1, s+b-1].  Cells
// where the reference reads face values it never wrote, or never writes the
// gradient, get NaN: their reconstructions reach no face flux the RHS uses.
//
// A block takes kGX x kGY cells and computes the velocities of them and their
// halos once, into LDS: in a pass per direction with the stencil's velocities
// per thread, five divisions a component, 1000 x 800 cells took 48 instead of
// 38 us.
constexpr int kGX = 32, kGY = 8;

template <int NF, int D, int WO, bool UNI>
__global__ __launch_bounds__(kGX *kGY) void k_visc_grad(ViscGradArgs g) {
    using Y = Sys<NF, D>;
    constexpr int P = (WO - 1) / 2;
    constexpr int CX = D == 2 ? kGX : kGX * kGY, CY = D == 2 ? kGY : 1; // cells of the tile
    constexpr int PY = D == 2 ? P : 0;
    constexpr int HX = CX + 2 * P, HY = CY + 2 * PY;
    __shared__ double su[D][HY][HX];
    const int tid = threadIdx.x;
    const int nyg = D == 2 ? g.s[1] + 1 + 2 * g.b : 1;
    const int x0 = (int)(blockIdx.x % g.ntile) * CX, y0 = (int)(blockIdx.x / g.ntile) * CY; // ghosted cell counts
    for (int e = tid; e < HX * HY; e += kGX * kGY) {
        const int r = e / HX, c = e % HX;
        const long o = min(max(x0 + c - P, 0), (int)g.nxg - 1) + g.nxg * (long)min(max(y0 + r - PY, 0), nyg - 1);
        double rho = 0.0;
#pragma unroll
        for (int f = 0; f < NF; ++f) rho = rho + g.q.v[f][o];
        rho = max_ref(rho, 1e-16);
#pragma unroll
        for (int d = 0; d < D; ++d) su[d][r][c] = g.q.v[Y::MOM + d][o] / rho;
    }
    __syncthreads();
    const int tx = tid % CX, ty = tid / CX, xg = x0 + tx, yg = y0 + ty;
    if (xg >= g.nxg || yg >= nyg) return;
    const long o = xg + g.nxg * (long)yg;
#pragma unroll
    for (int e = 0; e < D; ++e) {
        const int i = (e == 0 ? xg : yg) - g.b; // the cell's index along e
        const bool set = i >= -g.b + P && i <= g.s[e] + g.b - P && i >= -g.b + 1 && i <= g.s[e] + g.b - 1;
        double cf[kNCoef], inv = 0.0;
        if (set) {
#pragma unroll
            for (int q = 0; q < kNCoef; ++q) cf[q] = UNI ? g.ucf[e][q] : g.coef[e][(long)q * g.ncell[e] + (i + g.b)];
            inv = g.inv_dsg[e][i + g.b];
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
            double val = __builtin_nan("");
            if (set) {
                double st[WO], vl, vr;
#pragma unroll
                for (int r = 0; r < WO; ++r)
                    st[r] = e == 0 ? su[d][ty + PY][tx + r] : su[d][ty + r][tx + P];
                weno_cell<WO, double, true, true>(st, cf, g.eps, vl, vr);
                val = inv * (vr - vl);
            }
            g.grad[(long)(e * D + d) * g.ng + o] = val;
        }
    }
}

// x direction: one wave per 62 cells f0+1 .. f0+62 of row y (f0 = -1 +
// 62*tile).  Lane l converts stencil cells into LDS once, then reconstructs
// both faces of cell c = f0 + l (the smoothness indicators shared, as in the
// cell-parallel sweeps); face f = c takes its right state, the left-face
// value of cell c+1, from the next lane, and cell f+1 its upper face's fluxes
// the same way.  Bound by FP64 issue (1000 x 800 cells, two fluids, per-cell
// coefficients: 2470 vector instructions a wave, 1960 of them FP64).  With the
// faces' records stored for a finish kernel, and the gradients' face averages
// by another pass, the direction took 71 + 22 + 40 us instead of 90 together.
template <int NF, int D, int WO, bool UNI, bool WRF>
__global__ __launch_bounds__(64) void k_visc_x(ViscArgs a, SweepArgs s, int ntile) {
    using Y = Sys<NF, D>;
    constexpr int S = Y::S;
    constexpr int P = (WO - 1) / 2;
    constexpr int NS = 65 + 2 * P; // staged cells f0-P .. f0+64+P
    __shared__ double sp[S][NS];
    const int lane = threadIdx.x;
    const int tile = (int)(blockIdx.x % ntile);
    const int y = (int)(blockIdx.x / ntile);
    const int f0 = -1 + 62 * tile;
    const int hi = a.m + a.b; // last ghost cell
    for (int k = lane; k < NS; k += 64) {
        const int c = min(f0 - P + k, hi);
        const long o = goff(a, c, y);
        double cv[S], pv[S];
#pragma unroll
        for (int v = 0; v < S; ++v) cv[v] = a.q.v[v][o];
        cons_to_prim<NF, D>(cv, pv, a.eos);
#pragma unroll
        for (int v = 0; v < S; ++v) sp[v][k] = pv[v];
    }
    __syncthreads();
    const int c = min(f0 + lane, hi - P); // this lane's cell (clamped past the last face)
    double cf[kNCoef];
    cell_coef<UNI>(a, c, cf);
    // face averages of the gradient planes, reconstructed along x
    // (s_reconstruct_cell_boundary_values_visc_deriv, m_viscous.fpp:471-591)
    __shared__ double sg[WRF ? D * D : 1][64]; // rows only this lane reads back
    if constexpr (WRF) {
        const long o = goff(a, c, y);
        const int f = min(f0 + lane, a.m);
#pragma unroll 1
        for (int pl = 0; pl < D * D; ++pl) {
            const double *G = a.grad + (long)pl * a.ng + o;
            double st[WO], vl, vr;
#pragma unroll
            for (int r = 0; r < WO; ++r) st[r] = G[r - P];
            weno_cell<WO, double, true, true>(st, cf, a.eps, vl, vr);
            sg[pl][lane] = grad_average(a, f, a.m, vr, __shfl_down(vl, 1, 64));
        }
    }
    // one variable's registers at a time
    double ql[S], qr[S];
#pragma unroll
    for (int v = 0; v < S; ++v) {
        double st[WO], vl;
#pragma unroll
        for (int r = 0; r < WO; ++r) st[r] = sp[v][lane + r];
        weno_cell<WO, double, true, true>(st, cf, a.eps, vl, ql[v]);
        qr[v] = __shfl_down(vl, 1, 64);
        pin(ql[v], qr[v]);
    }
    // velocities of rows y-1 and y+1 of this lane's cell, then of the next
    // lane's (2D transverse gradients)
    double gt[2] = {0.0, 0.0};
    if constexpr (D == 2 && !WRF) {
        double um[2], up[2], um1[2], up1[2];
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            um[d] = cell_vel<NF, D>(a, c, y - 1, d);
            up[d] = cell_vel<NF, D>(a, c, y + 1, d);
        }
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            um1[d] = __shfl_down(um[d], 1, 64);
            up1[d] = __shfl_down(up[d], 1, 64);
        }
        const double dym = a.ccy[y + a.b] - a.ccy[y - 1 + a.b], dyp = a.ccy[y + 1 + a.b] - a.ccy[y + a.b];
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            const double u0 = sp[Y::MOM + d][lane + P], u1 = sp[Y::MOM + d][lane + P + 1];
            // four-point average of the one-sided y differences of cells
            // x+1 and x (dqR_prim_dy_n(1) at x, m_viscous.fpp:318-336)
            const double sum = (u1 - um1[d]) / dym + (up1[d] - u1) / dyp + (u0 - um[d]) / dym + (up[d] - u0) / dyp;
            gt[d] = 25e-2 * sum;
        }
    }
    const int f = min(f0 + lane, a.m); // (clamped past the last face)
    if (f == -1 && a.bc_beg == -4) {
#pragma unroll
        for (int v = 0; v < S; ++v) ql[v] = qr[v];
    }
    if (f == a.m && a.bc_end == -4) {
#pragma unroll
        for (int v = 0; v < S; ++v) qr[v] = ql[v];
    }
    double ax[2], ay[2];
    if constexpr (WRF) {
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            ax[d] = d < D ? sg[d][lane] : 0.0;
            ay[d] = d < D && D == 2 ? sg[D + d][lane] : 0.0;
        }
    } else {
        // one-sided x differences across the face (dqR_prim_dx_n(1) at x)
        double gxn[2] = {0.0, 0.0};
        const double dxf = a.ccx[f + 1 + a.b] - a.ccx[f + a.b];
#pragma unroll
        for (int d = 0; d < D; ++d) gxn[d] = (sp[Y::MOM + d][lane + P + 1] - sp[Y::MOM + d][lane + P]) / dxf;
        fd_averages<D, 0>(gxn, gt, ax, ay);
    }
    double flux[S], ustar, fs[D + 1];
    face_flux<NF, D, 0>(a, ql, qr, ax, ay, flux, ustar, fs);
    const double dus = __shfl_down(ustar, 1, 64) - ustar;
#pragma unroll
    for (int v = 0; v < S; ++v) flux[v] = flux[v] - __shfl_down(flux[v], 1, 64);
#pragma unroll
    for (int v = 0; v <= D; ++v) fs[v] = fs[v] - __shfl_down(fs[v], 1, 64);
    const int i = f0 + lane + 1;
    if (lane < 62 && i <= a.m) visc_finish<NF, D>(s, i, y, a.inv_ds[i], flux, dus, fs);
}

// y direction (2D), cell-parallel on an LDS tile: a block covers kYC
// x-columns by kYK cells along y, the K lanes of a column consecutive in the
// wave.  The primitive stencil rows of the tile (for finite-difference
// gradients with one x-halo column on each side) are converted once into LDS;
// thread (column, c) reconstructs both faces of cell f0+c one variable at a
// time (the WENO of the sweeps) and takes the state above its upper face from
// the next lane, the first K-1 lanes of each column solve their faces (HLLC,
// face Reynolds numbers, gradients, viscous flux), and after the faces' fluxes
// have replaced the tile in LDS the K-2 cells between them are finished with
// the threads along x.  (A thread marching along y with the stencil window in
// registers held 256 VGPRs and 72 AGPRs: one wave per SIMD.)  As in x, one
// kernel instead of three: 1000 x 800 cells, two fluids, 110 instead of 80 +
// 48 + 37 us.  The face states stay in registers: in LDS they halved the
// blocks per CU (136 us).  32 rows a tile are level with 16.
constexpr int kYC = 16; // x-columns per tile
constexpr int kYK = 16; // cells per column (faces: kYK - 1, finished cells: kYK - 2)

template <int NF, int WO, bool UNI, bool WRF>
__global__ __launch_bounds__(kYC *kYK) void k_visc_y(ViscArgs a, SweepArgs s, int nxb) {
    constexpr int D = 2;
    using Y = Sys<NF, D>;
    constexpr int S = Y::S;
    constexpr int P = (WO - 1) / 2;
    constexpr int R = kYK + 2 * P;  // stencil rows f0-P .. f0+K-1+P
    constexpr int XH = WRF ? 0 : 1; // x-halo columns on each side
    constexpr int XC = kYC + 2 * XH;
    // stencil rows of each column contiguous (odd pitch R + 1): the lanes of
    // a column read consecutive entries
    using Tile = double[XC][R + 1];
    // then the S fluxes, the contact velocity and the viscous fluxes of face
    // f0+c+1/2 of column col, with an odd pitch for the finish along x
    using Face = double[kYC][kYK + 1];
    constexpr int NT = S * sizeof(Tile) / 8, NF_ = (S + 2 + D) * sizeof(Face) / 8;
    __shared__ double sh[NT > NF_ ? NT : NF_];
    Tile *sp = reinterpret_cast<Tile *>(sh);
    Face *sf = reinterpret_cast<Face *>(sh);
    const int tid = threadIdx.x;
    const int col = tid / kYK, c = tid % kYK;
    const int x0 = (int)(blockIdx.x % nxb) * kYC;
    const int f0 = -1 + (kYK - 2) * (int)(blockIdx.x / nxb);
    const int hx = a.m + a.b, hy = a.n + a.b; // last ghost cells
    const int x = x0 + col;
    const int f = f0 + c; // this lane's cell, and the face above it
    double cf[kNCoef];
    cell_coef<UNI>(a, min(f, hy - P), cf);
    // face averages of the gradient planes, reconstructed along y
    __shared__ double sg[WRF ? D * D : 1][kYC * kYK]; // slots only their own thread reads back
    if constexpr (WRF) {
        static_assert(S >= D * D, "the gradient planes fit in the tile");
        for (int e = tid; e < R * kYC; e += kYC * kYK) {
            const int r = e / kYC, xc = e % kYC;
            const long o = goff(a, min(x0 + xc, hx), min(f0 - P + r, hy));
#pragma unroll
            for (int pl = 0; pl < D * D; ++pl) sp[pl][xc][r] = a.grad[(long)pl * a.ng + o];
        }
        __syncthreads();
#pragma unroll 1
        for (int pl = 0; pl < D * D; ++pl) {
            double st[WO], vl, vr;
#pragma unroll
            for (int r = 0; r < WO; ++r) st[r] = sp[pl][col][c + r];
            weno_cell<WO, double, true, true>(st, cf, a.eps, vl, vr);
            sg[pl][tid] = grad_average(a, f, a.n, vr, __shfl_down(vl, 1, 64));
        }
        __syncthreads();
    }
    for (int e = tid; e < R * XC; e += kYC * kYK) {
        const int r = e / XC, xc = e % XC;
        const long o = goff(a, min(x0 - XH + xc, hx), min(f0 - P + r, hy));
        double cv[S], pv[S];
#pragma unroll
        for (int v = 0; v < S; ++v) cv[v] = a.q.v[v][o];
        cons_to_prim<NF, D>(cv, pv, a.eos);
#pragma unroll
        for (int v = 0; v < S; ++v) sp[v][xc][r] = pv[v];
    }
    __syncthreads();
    // one variable's registers at a time; lane c+1 of the same column holds
    // cell f0+c+1 (the last lane's value is not used)
    double ql[S], qr[S];
#pragma unroll
    for (int v = 0; v < S; ++v) {
        double st[WO], vl;
#pragma unroll
        for (int r = 0; r < WO; ++r) st[r] = sp[v][col + XH][c + r];
        weno_cell<WO, double, true, true>(st, cf, a.eps, vl, ql[v]);
        qr[v] = __shfl_down(vl, 1, 64);
        pin(ql[v], qr[v]);
    }
    const bool face = c < kYK - 1 && x <= a.m && f <= a.n;
    double flux[S], ustar, fs[D + 1];
    if (face) {
        if (f == -1 && a.bc_beg == -4) {
#pragma unroll
            for (int v = 0; v < S; ++v) ql[v] = qr[v];
        }
        if (f == a.n && a.bc_end == -4) {
#pragma unroll
            for (int v = 0; v < S; ++v) qr[v] = ql[v];
        }
        double ax[2], ay[2];
        if constexpr (WRF) {
#pragma unroll
            for (int d = 0; d < 2; ++d) ax[d] = sg[d][tid], ay[d] = sg[D + d][tid];
        } else {
            // velocities of cells (x-1 .. x+1, f) and (x-1 .. x+1, f+1)
            const int r0 = c + P, r1 = c + P + 1;
            const double dyf = a.ccy[f + 1 + a.b] - a.ccy[f + a.b];
            const double dxm = a.ccx[x + a.b] - a.ccx[x - 1 + a.b], dxp = a.ccx[x + 1 + a.b] - a.ccx[x + a.b];
            double gxn[2], gt[2];
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                const double(*u)[R + 1] = &sp[Y::MOM + d][col];
                const double uo = u[1][r0], uw = u[0][r0], ue = u[2 * XH][r0];
                const double no = u[1][r1], nw = u[0][r1], ne = u[2 * XH][r1];
                gxn[d] = (no - uo) / dyf;
                // four-point average of the one-sided x differences of rows f+1
                // and f (dqR_prim_dx_n(2) at f, m_viscous.fpp:285-315)
                const double sum = (no - nw) / dxm + (ne - no) / dxp + (uo - uw) / dxm + (ue - uo) / dxp;
                gt[d] = 25e-2 * sum;
            }
            fd_averages<D, 1>(gxn, gt, ax, ay);
        }
        face_flux<NF, D, 1>(a, ql, qr, ax, ay, flux, ustar, fs);
    }
    __syncthreads();
    if (face) {
#pragma unroll
        for (int v = 0; v < S; ++v) sf[v][col][c] = flux[v];
        sf[S][col][c] = ustar;
#pragma unroll
        for (int v = 0; v <= D; ++v) sf[S + 1 + v][col][c] = fs[v];
    }
    __syncthreads();
    const int fx = tid % kYC, r = tid / kYC, i = x0 + fx, j = f0 + 1 + r;
    if (r >= kYK - 2 || i > a.m || j > a.n) return;
    double d[S], dv[D + 1];
#pragma unroll
    for (int v = 0; v < S; ++v) d[v] = sf[v][fx][r] - sf[v][fx][r + 1];
#pragma unroll
    for (int v = 0; v <= D; ++v) dv[v] = sf[S + 1 + v][fx][r] - sf[S + 1 + v][fx][r + 1];
    visc_finish<NF, D>(s, i, j, a.inv_ds[j], d, sf[S][fx][r + 1] - sf[S][fx][r], dv);
}

template <int NF, int D, int DIR, int WO, bool UNI, bool WRF>
void launch_dir_u(const ViscArgs &a, const SweepArgs &sa, hipStream_t st) {
    if constexpr (DIR == 0) {
        const int ntile = (a.m + 1 + 61) / 62;
        hipLaunchKernelGGL((k_visc_x<NF, D, WO, UNI, WRF>), dim3((unsigned)((long)ntile * (a.n + 1))), dim3(64), 0, st,
                           a, sa, ntile);
    } else {
        const int nxb = (a.m + 1 + kYC - 1) / kYC;
        const int ntile = (a.n + 1 + kYK - 3) / (kYK - 2);
        hipLaunchKernelGGL((k_visc_y<NF, WO, UNI, WRF>), dim3((unsigned)((long)nxb * ntile)), dim3(kYC * kYK), 0, st,
                           a, sa, nxb);
    }
}

template <int NF, int D, int DIR, int WO>
int launch_order(const ViscArgs &a, const SweepArgs &sa, hipStream_t st) {
    if (a.wrf) {
        if (a.uniform) launch_dir_u<NF, D, DIR, WO, true, true>(a, sa, st);
        else launch_dir_u<NF, D, DIR, WO, false, true>(a, sa, st);
    } else {
        if (a.uniform) launch_dir_u<NF, D, DIR, WO, true, false>(a, sa, st);
        else launch_dir_u<NF, D, DIR, WO, false, false>(a, sa, st);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int NF, int D, int DIR>
int launch_dir(int weno_order, const ViscArgs &a, const SweepArgs &sa, hipStream_t st) {
    switch (weno_order) {
    case 1: return launch_order<NF, D, DIR, 1>(a, sa, st);
    case 3: return launch_order<NF, D, DIR, 3>(a, sa, st);
    case 5: return launch_order<NF, D, DIR, 5>(a, sa, st);
    default: return -1;
    }
}

template <int NF>
int launch_nf(int D, int dir, int weno_order, const ViscArgs &a, const SweepArgs &sa, hipStream_t st) {
    if (D == 1 && dir == 0) return launch_dir<NF, 1, 0>(weno_order, a, sa, st);
    if (D == 2 && dir == 0) return launch_dir<NF, 2, 0>(weno_order, a, sa, st);
    if (D == 2 && dir == 1) return launch_dir<NF, 2, 1>(weno_order, a, sa, st);
    return -1;
}

template <int NF, int D>
int launch_grad(int weno_order, ViscGradArgs g, hipStream_t st) {
    const int cx = D == 2 ? kGX : kGX * kGY, cy = D == 2 ? kGY : 1;
    const int nyg = D == 2 ? g.s[1] + 1 + 2 * g.b : 1;
    g.ntile = (int)((g.nxg + cx - 1) / cx);
    const dim3 grid((unsigned)((long)g.ntile * ((nyg + cy - 1) / cy))), block(kGX * kGY);
    const bool u = g.uniform != 0;
    switch (weno_order) {
    case 1: hipLaunchKernelGGL((k_visc_grad<NF, D, 1, false>), grid, block, 0, st, g); break;
    case 3:
        if (u) hipLaunchKernelGGL((k_visc_grad<NF, D, 3, true>), grid, block, 0, st, g);
        else hipLaunchKernelGGL((k_visc_grad<NF, D, 3, false>), grid, block, 0, st, g);
        break;
    case 5:
        if (u) hipLaunchKernelGGL((k_visc_grad<NF, D, 5, true>), grid, block, 0, st, g);
        else hipLaunchKernelGGL((k_visc_grad<NF, D, 5, false>), grid, block, 0, st, g);
        break;
    default: return -1;
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int NF>
int launch_grad_nf(int D, int weno_order, const ViscGradArgs &g, hipStream_t st) {
    if (D == 1) return launch_grad<NF, 1>(weno_order, g, st);
    if (D == 2) return launch_grad<NF, 2>(weno_order, g, st);
    return -1;
}

} // namespace

int launch_visc_grad(int nf, int D, int weno_order, const ViscGradArgs &g, hipStream_t st) {
    switch (nf) {
    case 1: return launch_grad_nf<1>(D, weno_order, g, st);
    case 2: return launch_grad_nf<2>(D, weno_order, g, st);
    case 3: return launch_grad_nf<3>(D, weno_order, g, st);
    case 4: return launch_grad_nf<4>(D, weno_order, g, st);
    default: return -1;
    }
}

int launch_viscous(int nf, int D, int dir, int weno_order, const ViscArgs &a, const SweepArgs &sa,
                   hipStream_t st) {
    switch (nf) {
    case 1: return launch_nf<1>(D, dir, weno_order, a, sa, st);
    case 2: return launch_nf<2>(D, dir, weno_order, a, sa, st);
    case 3: return launch_nf<3>(D, dir, weno_order, a, sa, st);
    case 4: return launch_nf<4>(D, dir, weno_order, a, sa, st);
    default: return -1;
    }
}

} // namespace mfc
