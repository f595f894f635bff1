// mfc_rows.hpp -- x sweep of row after row by the same columns (FP64, WENO5,
// unequal widths, 2D and 3D, one to three fluids).
#pragma once

#include "mfc_sweep.hpp"

namespace mfc {

constexpr int kRowsCells = 58; // cells a wave finishes per row
constexpr int kRowsMaxFluids = 3;

inline namespace MFC_FORM {

// x sweep of 64 neighbouring columns, a.chunk rows along y in turn.  Lane l of a
// wave holds entry 58 set + l of the rows of the planes set end to end, a.rl
// entries each (three x ghost cells at either end): both faces of its cell (its
// 27 coefficients are loaded once and stay in registers), the right state of a
// face from the next lane, the lower flux of a cell from the one before; lanes
// 3 .. 60 finish their cell where it is an interior one.  The next row's cells
// are loaded during this row's arithmetic.
//
// k_sweep_x reads the coefficients of both cells of a face per row, 54 loads
// beside the S variables', and computes the smoothness indicators of each cell
// twice, since a lane with one cell's both faces lost a wave of occupancy.
// Here the loads are shared by the rows and two waves per SIMD are enough (142
// to 229 VGPRs; at three the coefficients spill): 180 x 130 x 90 cells, three
// fluids, contracted 0.201 -> 0.151 ms per launch, 256 x 200 x 160 0.827 ->
// 0.538, plain 700 x 700, two fluids 0.044 -> 0.037 ms.
template <int NF, int D>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_rows_x(const SweepArgs a) {
    using Y = Sys<NF, D>;
    constexpr int S = Y::S;
    constexpr int FM = finish_modes<D, true, double, false>();
    __shared__ double sp[S][64];
    const long bid = xcd_logical_block(blockIdx.x, a.nblocks);
    const int set = (int)(bid % a.ntile), lane = threadIdx.x;
    const int r0 = (int)(bid / a.ntile) * a.chunk, r1 = min(r0 + a.chunk, a.n + 1);
    const int g0 = set * kRowsCells, t0 = g0 / a.rl;
    int t = (g0 + lane) / a.rl, x = g0 + lane - t * a.rl - 3;
    if (t > a.p) t = a.p, x = a.m + 3;
    double cf[kNCoef];
    load_coef<double, 5, false>(a, min(max(x, -1), a.m + 1), cf);
    const double eps = a.eps;
    const bool fin_lane = lane >= 3 && lane <= 60 && x >= 0 && x <= a.m;
    const int xc = min(max(x, 0), a.m);
    // lane parts of the offsets from row j of plane t0
    const unsigned own = (unsigned)(t - t0) * (unsigned)(a.nxg * a.nyg) + (unsigned)(x + 3);
    const unsigned cell = (unsigned)(t - t0) * (unsigned)(a.nxg * a.nyg) + (unsigned)xc;
    const unsigned rcell = (unsigned)(t - t0) * (unsigned)((a.m + 1) * (a.n + 1)) + (unsigned)xc;
    const double inv = a.inv_ds[xc];
    const int l0 = min(max(lane - 2, 0), 59); // first stencil entry
    double cv[S];
    auto load = [&](int j) {
        const Off o{ghost_off(a, -3, j, t0), own};
#pragma unroll
        for (int v = 0; v < S; ++v) cv[v] = el(a.qin.v[v], o);
    };
    load(r0);
#pragma unroll 1
    for (int j = r0; j < r1; ++j) {
        {
            double pr[S];
            cons_to_prim<NF, D>(cv, pr, a.eos);
#pragma unroll
            for (int v = 0; v < S; ++v) sp[v][lane] = pr[v];
        }
        load(min(j + 1, r1 - 1));
        wave_lds_sync();
        const Off go{ghost_off(a, 0, j, t0), cell}, ro{interior_off(a, 0, j, t0), rcell};
        double qL[S], qR[S], f[S], us;
#pragma unroll
        for (int v = 0; v < S; ++v) {
            double st[5], vl;
#pragma unroll
            for (int w = 0; w < 5; ++w) st[w] = sp[v][l0 + w];
            weno_both<5, double, false>(st, cf, eps, vl, qL[v], CanonK());
            qR[v] = __shfl_down(vl, 1, 64);
            asm volatile("" : "+v"(qL[v]), "+v"(qR[v]));
        }
        wave_lds_sync();
        if (x == -1 && a.bc_beg == -4) {
#pragma unroll
            for (int v = 0; v < S; ++v) qL[v] = qR[v];
        }
        if (x == a.m && a.bc_end == -4) {
#pragma unroll
            for (int v = 0; v < S; ++v) qR[v] = qL[v];
        }
        hllc_face<NF, D, 0, double>(qL, qR, a.eos, f, us);
        double fm[S];
#pragma unroll
        for (int v = 0; v < S; ++v) fm[v] = __shfl_up(f[v], 1, 64);
        const double usm = __shfl_up(us, 1, 64);
        if (fin_lane) {
            FinishIn<S> fin;
            finish_load<NF, D, FM>(a, go, ro, fin);
            finish_cell<NF, D, double, FM, false>(a, go, ro, inv, fm, f, usm, us, fin, a.base_lo, a.base_hi, x, j);
        }
    }
}

} // namespace MFC_FORM
} // namespace mfc
