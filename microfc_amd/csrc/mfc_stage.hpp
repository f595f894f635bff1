// mfc_stage.hpp -- one kernel for a whole RK stage of a small 1D or 2D case
// (plain and contracted FP64, WENO5, one or two fluids).
#pragma once

#include "mfc_sweep.hpp"

namespace mfc {

// Tile of k_stage: kStageX x kStageY cells in 2D, kStageX1 cells in 1D.
constexpr int kStageX = 16, kStageY = 10, kStageX1 = 62;
constexpr int stage_cells_x(int D) { return D == 2 ? kStageX : kStageX1; }
constexpr int stage_cells_y(int D) { return D == 2 ? kStageY : 1; }
// Waves of the cells (with the end cells) of the x and of the y direction,
// groups of waves that share the variables, and threads.
constexpr int stage_waves_x(int D) { return ((stage_cells_x(D) + 2) * stage_cells_y(D) + 63) / 64; }
constexpr int stage_waves_y(int D) { return D == 2 ? (kStageX * (kStageY + 2) + 63) / 64 : 0; }
constexpr int stage_groups(int NF, int D) { return D == 2 ? 2 : 2 * NF + D + 1; }
constexpr int stage_threads(int NF, int D) { return 64 * (stage_waves_x(D) + stage_waves_y(D)) * stage_groups(NF, D); }

template <int NF, int D> struct StageTile {
    static constexpr int S = 2 * NF + D + 1;
    static constexpr int P = 2, H = P + 1; // stencil half width, staged halo
    static constexpr int CX = stage_cells_x(D), CY = stage_cells_y(D);
    static constexpr int NX = CX + 2 * H, NY = D == 2 ? CY + 2 * H : 1; // staged cells (without the corners)
    static constexpr int PX = NX | 1;                                  // their row pitch in LDS
    static constexpr int WX = stage_waves_x(D), WY = stage_waves_y(D), SLOTS = 64 * (WX + WY);
    static constexpr int G = stage_groups(NF, D), T = stage_threads(NF, D), WAVES = T / 64;
    static constexpr int WC = (CX * CY + 63) / 64; // waves of the tile's cells
    static constexpr int ROUNDS = (S * WC + WAVES - 1) / WAVES; // finish: a wave takes 64 cells of one variable
};

inline namespace MFC_FORM {

// Stores variable v (value r) of cell (i, j) into the ghost cells that copy
// it, as store_ghosts.
template <int D>
__device__ __forceinline__ void store_ghosts_of(const SweepArgs &a, double *q, int i, int j, bool mx, bool my, double r) {
    bool edge = i < a.b || i > a.m - a.b;
    if constexpr (D > 1) edge = edge || j < a.b || j > a.n - a.b;
    if (!edge) return;
    const GhostSet none{0, 0, 0, 0, false, false};
    const GhostSet ex = ghosts_of(i, a.m, a.bcs[0], a.b);
    const GhostSet ey = D > 1 ? ghosts_of(j, a.n, a.bcs[1], a.b) : none;
    auto copy = [](const GhostSet &e, int c, int own, bool &flip) {
        flip = c == 0 ? false : c <= e.n0 ? e.flip0 : e.flip1;
        return c == 0 ? own : c <= e.n0 ? e.g0 + c - 1 : e.g1 + c - 1 - e.n0;
    };
#pragma unroll 1
    for (int cj = 0; cj <= ey.n0 + ey.n1; ++cj) {
        bool fj, fi;
        const int gj = copy(ey, cj, j, fj);
#pragma unroll 1
        for (int ci = cj == 0 ? 1 : 0; ci <= ex.n0 + ex.n1; ++ci) {
            const int gi = copy(ex, ci, i, fi);
            q[ghost_off(a, gi, gj, 0)] = (mx && fi) || (my && fj) ? -r : r;
        }
    }
}

// One RK stage (rk, from qin and qbase into qout) of a 1D or 2D case, every
// direction at once:
//  1. the tile's cells and their halo are staged (cons->prim) in LDS, ghost
//     cells from the interior cells they copy, and the finish's inputs are
//     loaded;
//  2. the waves share the cells of both directions and, in G groups, the
//     variables: each reconstructs both faces of its cells;
//  3. one wave per 64 faces solves them (HLLC), x and y faces side by side;
//  4. a wave finishes 64 cells of one variable: the directions' flux
//     differences and alpha*div(u) sources in the reference's order (in the
//     plain form bitwise the separate sweeps), then the RK stage; and with
//     a.ghosts fills the input's ghost cells.
// For grids that leave most of the chip idle, where a stage is the latency of
// its kernels: the ghost fill and the separate x and y sweeps, one wave per 62
// cells with every variable in turn, took 3.7 + 10.5 + 10.4 us on 200 x 150
// cells, this 15.8 (adaptive RK3 step 105 -> 76 us); 1000 cells 7.0 -> 5.8 us.  By its
// own clock (2D, per-cell coefficients): loads 2.1 us, conversion 0.6,
// reconstruction 4.4, faces 1.9, finish 1.2.  Coefficients loaded per wave
// instead of per block cost 1.4 us more.
template <int NF, int D, int UNI>
__global__ __launch_bounds__(stage_threads(NF, D)) void k_stage(const SweepArgs a) {
    using L = StageTile<NF, D>;
    using Y = Sys<NF, D>;
    constexpr int S = Y::S, P = L::P, H = L::H, CX = L::CX, CY = L::CY, T = L::T, NX = L::NX, PX = L::PX;
    using Row = double[L::NY][PX];
    using Slots = double[L::SLOTS];
    constexpr int NSP = S * sizeof(Row) / 8, NF_ = (S + 1) * L::SLOTS;
    __shared__ double lds[NSP > NF_ ? NSP : NF_]; // staged primitives, then the face fluxes and contact velocities
    __shared__ double up[S][L::SLOTS], lo[S][L::SLOTS]; // values at the upper and lower face of a slot's cell
    constexpr int NC = CX + 2 + (D == 2 ? CY + 2 : 0);
    __shared__ double cs[UNI ? 1 : kNCoef][UNI ? 1 : NC];
    Row *sp = reinterpret_cast<Row *>(lds);
    Slots *fl = reinterpret_cast<Slots *>(lds);
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int x0 = (int)(blockIdx.x % (unsigned)a.ntile) * CX, y0 = (int)(blockIdx.x / (unsigned)a.ntile) * CY;

    // 1. every load of the kernel before the first value is used: the staged
    // cells (one per thread), the coefficients of the tile's cells in x, then
    // in y, and the finish's inputs
    constexpr int ROWC = NX * CY, NST = ROWC + (D == 2 ? 2 * H * CX : 0);
    static_assert(NST <= T, "one staged cell per thread");
    int ii, jj; // staged column and row
    if (tid < ROWC) {
        ii = tid % NX;
        jj = tid / NX + (D == 2 ? H : 0);
    } else {
        const int h = tid - ROWC, r = h / CX;
        ii = h % CX + H;
        jj = r < H ? r : min(r + CY, L::NY - 1); // (past the last staged cell: not stored)
    }
    double cv[S];
    bool mx = false, my = false; // mirrored
    {
        const int i = bc_source(a.bcs[0][0], a.bcs[0][1], a.m, min(x0 - H + ii, a.m + a.b), mx);
        const int j = D == 2 ? bc_source(a.bcs[1][0], a.bcs[1][1], a.n, min(y0 - H + jj, a.n + a.b), my) : 0;
        const long o = ghost_off(a, i, j, 0);
#pragma unroll
        for (int v = 0; v < S; ++v) cv[v] = a.qin.v[v][o];
    }
    constexpr int NCF = UNI ? 0 : (kNCoef * NC + T - 1) / T;
    double cl[NCF + 1];
#pragma unroll
    for (int t = 0; t < NCF; ++t) {
        const int e = min(tid + t * T, kNCoef * NC - 1), q = e / NC, c = e % NC;
        const bool y = c >= CX + 2;
        const double *p = y ? a.coef2 + (long)q * a.ncell2 + (min(y0 - 1 + c - (CX + 2), a.n + 1) + a.b)
                            : a.coef + (long)q * a.ncell + (min(x0 - 1 + c, a.m + 1) + a.b);
        cl[t] = *p;
    }
    double base[L::ROUNDS], in[L::ROUNDS], ix[L::ROUNDS], iy[L::ROUNDS];
#pragma unroll
    for (int t = 0; t < L::ROUNDS; ++t) {
        const int u = w + t * L::WAVES, v = min(u / L::WC, S - 1), cell = min((u % L::WC) * 64 + lane, CX * CY - 1);
        const int i = min(x0 + cell % CX, a.m), j = min(y0 + cell / CX, a.n);
        const long o = ghost_off(a, i, j, 0);
        base[t] = a.qbase.v[v][o];
        in[t] = a.qin.v[v][o];
        ix[t] = a.inv_ds[i];
        iy[t] = D == 2 ? a.inv_ds2[j] : 0.0;
    }
    if (tid < NST) {
        double pv[S];
        if (mx) cv[Y::MOM] = -cv[Y::MOM];
        if constexpr (D == 2)
            if (my) cv[Y::MOM + 1] = -cv[Y::MOM + 1];
        cons_to_prim<NF, D>(cv, pv, a.eos);
#pragma unroll
        for (int v = 0; v < S; ++v) sp[v][jj][ii] = pv[v];
    }
#pragma unroll
    for (int t = 0; t < NCF; ++t)
        if (const int e = tid + t * T; e < kNCoef * NC) cs[UNI ? 0 : e / NC][UNI ? 0 : e % NC] = cl[t];
    __syncthreads();

    // 2.
    {
        const int g = w / (L::WX + L::WY), ws = w % (L::WX + L::WY), slot = ws * 64 + lane;
        const bool isx = D == 1 || ws < L::WX;
        const int st = isx ? slot : slot - L::WX * 64; // cell of the direction: rows of CX + 2, or columns of CY + 2
        const int wi = isx ? st % (CX + 2) : st % CX, wj = isx ? min(st / (CX + 2), CY - 1) : min(st / CX, CY + 1);
        const double *uni = isx ? a.ucf : a.ucf2;
        const int cc = isx ? wi : CX + 2 + wj;
        double cf[kNCoef];
#pragma unroll
        for (int q = 0; q < kNCoef; ++q) cf[q] = UNI ? uni[q] : cs[UNI ? 0 : q][UNI ? 0 : cc];
        // staged row and column, and the pitch of the direction
        const int ii = isx ? wi + H - 1 : wi + H, jj = D == 1 ? 0 : isx ? wj + H : wj + H - 1;
        const int pitch = isx ? 1 : PX;
        const double eps = a.eps;
#pragma unroll 1
        for (int v = g; v < S; v += L::G) {
            const double *q = &sp[v][jj][ii] - P * pitch;
            double sv[2 * P + 1];
#pragma unroll
            for (int r = 0; r <= 2 * P; ++r) sv[r] = q[r * pitch];
            weno_both<5, double, UNI>(sv, cf, eps, lo[v][slot], up[v][slot], CanonK());
        }
    }
    __syncthreads();

    // 3. (the staged primitives are dead)
    auto solve = [&](auto dir, int slot, int next, int to, int f, int s, int bc0, int bc1) {
        constexpr int DIR = decltype(dir)::value;
        double ql[S], qr[S], flux[S], us;
#pragma unroll
        for (int v = 0; v < S; ++v) {
            ql[v] = up[v][slot];
            qr[v] = lo[v][next];
        }
        if (f == -1 && bc0 == -4) {
#pragma unroll
            for (int v = 0; v < S; ++v) ql[v] = qr[v];
        }
        if (f == s && bc1 == -4) {
#pragma unroll
            for (int v = 0; v < S; ++v) qr[v] = ql[v];
        }
        hllc_face<NF, D, DIR, double>(ql, qr, a.eos, flux, us);
#pragma unroll
        for (int v = 0; v < S; ++v) fl[v][to] = flux[v];
        fl[S][to] = us;
    };
    constexpr int FX = CX + 1, WFX = (FX * CY + 63) / 64;
    static_assert(WFX <= L::WX && (D == 1 || (CX * (CY + 1) + 63) / 64 <= L::WY), "faces fit in the cells' slots");
    if (w < WFX) {
        const int t = w * 64 + lane, fx = t % FX, row = t / FX, f = x0 - 1 + fx;
        if (row < CY && f <= a.m && y0 + row <= a.n)
            solve(std::integral_constant<int, 0>{}, row * (CX + 2) + fx, row * (CX + 2) + fx + 1, t, f, a.m, a.bc_beg,
                  a.bc_end);
    } else if constexpr (D == 2) {
        const int t = (w - WFX) * 64 + lane, col = t % CX, fy = t / CX, f = y0 - 1 + fy;
        if (fy <= CY && f <= a.n && x0 + col <= a.m)
            solve(std::integral_constant<int, 1>{}, L::WX * 64 + t, L::WX * 64 + t + CX, L::WX * 64 + t, f, a.n, a.bc2_beg,
                  a.bc2_end);
    }
    __syncthreads();

    // 4.
#pragma unroll
    for (int t = 0; t < L::ROUNDS; ++t) {
        const int u = w + t * L::WAVES, v = u / L::WC, cell = (u % L::WC) * 64 + lane;
        const int col = cell % CX, row = cell / CX, i = x0 + col, j = y0 + row;
        if (v >= S || cell >= CX * CY || i > a.m || j > a.n) continue;
        const int fx = row * FX + col, fy = L::WX * 64 + row * CX + col;
        double r = ix[t] * (fl[v][fx] - fl[v][fx + 1]);
        if (v >= Y::ADV) r = r + ix[t] * in[t] * (fl[S][fx + 1] - fl[S][fx]);
        if constexpr (D == 2) {
            r = r + iy[t] * (fl[v][fy] - fl[v][fy + CX]);
            if (v >= Y::ADV) r = r + iy[t] * in[t] * (fl[S][fy + CX] - fl[S][fy]);
        }
        FinishIn<1> f;
        f.base[0] = base[t];
        f.in[0] = in[t];
        double o;
        rk_combine<1>(a, f, &r, &o);
        a.qout.v[v][ghost_off(a, i, j, 0)] = o;
        if (a.ghosts) store_ghosts_of<D>(a, a.qin.v[v], i, j, v == Y::MOM, D == 2 && v == Y::MOM + 1, in[t]);
    }
}

} // namespace MFC_FORM
} // namespace mfc
