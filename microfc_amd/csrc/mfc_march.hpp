// mfc_march.hpp -- marching sweeps of large WENO5 cases, one to three fluids.
//
// A wave owns 64 neighbouring columns of cells and walks them along y or z
// row by row, so a row is converted to primitive once, each face of the
// marching direction is reconstructed and solved once (its lower flux is
// kept for the next row), and no lane waits for another wave:
//   * z march (MD = 2), and the y march alone (MD = 1, three fluids): every
//     lane's cell is finished;
//   * y march with the x faces of each row (WX): the lanes are consecutive
//     entries of the rows of the outer index set end to end, each row with
//     its three x ghost cells on either side; lanes 1 .. 62 finish their cell
//     where it is an interior one.  x stencils, face states and fluxes move
//     between lanes as in k_sweep_x.
// The last three primitive rows stay in an LDS ring private to the wave; the
// far end of the five-row stencil is kept in registers when its entry is
// overwritten, the current row until the end of its pass.  The next row's
// loads are in flight during the arithmetic of this one.
//
// What bounds it.  The tile kernels are bound by VALU issue (k_sweep_xy 77 %
// busy at 512^3, contracted form) and repeat work at their edges: k_sweep_xy
// converts 720 cells and solves 512 + 448 faces for 420 finished cells,
// k_sweep_tc 320 and 256 for 224.  A march converts and solves once per cell
// and direction, plus 2 of 64 lanes, 6 entries per row of x cells and about
// three rows per chunk: 2.92e9 instead of 3.59e9 VALU instructions (x and y)
// and 1.41e9 instead of 1.85e9 (z) per launch at 512^3, 8.35 -> 7.35 and 5.45
// -> 4.70 ms.  The z march then runs at the memory's rate (23 GB per launch,
// 4.8 TB/s, as a large copy); the x and y march (30 GB, 4.1 TB/s) at 75 % VALU
// busy, its two waves per SIMD waiting on LDS and memory for the rest.
//
// With three fluids the state of the x faces no longer fits beside the march's
// (the ring takes 15 KB a wave, the z march 176 to 224 VGPRs): x keeps its
// sweep, y and z march on their own.  180 x 130 x 90 stretched cells,
// contracted: y 0.203 -> 0.130, z 0.183 -> 0.118 ms per launch.
#pragma once

#include "mfc_sweep.hpp"

namespace mfc {

constexpr int kMarchCellsXY = 62, kMarchCellsZ = 64; // cells a wave can finish per row
constexpr int kMarchHaloXY = 3;                      // x ghost cells per row end in the entry order
constexpr int kMarchMaxFluidsXY = 2, kMarchMaxFluidsZ = 3;

inline namespace MFC_FORM {

// A table entry that is the same for the whole wave, read through the scalar
// cache (the tables are written by the host before any launch).
__device__ __forceinline__ double uniform_load(const double *p, long i) {
    return reinterpret_cast<const __attribute__((address_space(4))) double *>(reinterpret_cast<unsigned long>(p))[i];
}

// The kernel's arguments (its only parameter, so at the start of the kernarg
// segment), read again through the scalar cache.  Inside the row loop the
// pointers and coefficients of a phase are taken from here: kept live across
// the whole loop they overflow the scalar registers, and pointers advanced
// per row the vector registers too (456 bytes of scratch per lane).
__device__ __forceinline__ const SweepArgs &fresh_args() {
    unsigned long p = reinterpret_cast<unsigned long>(__builtin_amdgcn_kernarg_segment_ptr());
    asm volatile("" : "+s"(p));
    return *(const SweepArgs *)reinterpret_cast<const __attribute__((address_space(4))) SweepArgs *>(p);
}
// Values finished here.  Without it the arithmetic of a value that is used
// only after the next branch is sunk past it, with every variable's
// intermediates live until then (700 bytes of scratch per lane).
template <int N, typename R>
__device__ __forceinline__ void hold(R (&v)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(v[i]));
}

// Operands of the finish of one cell: first the rhs (3D: the sums begin in
// the z march, or in the plain form in the x and y march) and the RK base
// (of the variables lo .. hi-1 in a spread stage) ...  Every lane loads, from
// clamped cells where it has none to finish: loads under a branch were
// spilled as they arrived.
template <int NF, int D, bool RHS, int M>
__device__ __forceinline__ void march_load_acc(const SweepArgs &a, const SweepArgs &base, Off go, Off ro, int lo, int hi,
                                               FinishIn<Sys<NF, D>::S> &f) {
    constexpr int S = Sys<NF, D>::S;
    if constexpr (RHS) {
#pragma unroll
        for (int v = 0; v < S; ++v) f.rhs[v] = el(a.rhs.v[v], ro);
    }
    if (M != kModesAll && a.fold && a.cb != 0.0) {
#pragma unroll
        for (int v = 0; v < S; ++v)
            if (v >= lo && v < hi) f.base[v] = el(base.qbase.v[v], go);
    }
}
// ... and the stage input.  In FP64 its partial densities and volume
// fractions are primitive variables too (march_prim_in), and the x and y
// march keeps momentum and energy in LDS; otherwise they are read again
// where an RK stage can use them.
template <int NF, int D, typename R, bool WX, int M>
__device__ __forceinline__ void march_load_in(const SweepArgs &a, Off go, FinishIn<Sys<NF, D>::S> &f) {
    using Y = Sys<NF, D>;
    constexpr int S = Y::S;
    constexpr bool RING = sizeof(R) == 8, RK = M != kModesFoldFirst;
#pragma unroll
    for (int v = 0; v < S; ++v) {
        const bool same = v < NF || v >= Y::ADV;
        if (same ? !RING && (RK || v >= Y::ADV) : RK && !(RING && WX)) f.in[v] = el(a.qin.v[v], go);
    }
    if (M == kModesAll && a.rk != kRkNone && !a.base_is_in) {
#pragma unroll
        for (int v = 0; v < S; ++v) f.base[v] = el(a.qbase.v[v], go);
    }
}
template <int NF, int D, typename R, int M>
__device__ __forceinline__ void march_prim_in(const SweepArgs &a, const R *prim, FinishIn<Sys<NF, D>::S> &f) {
    using Y = Sys<NF, D>;
    constexpr int S = Y::S;
    if (sizeof(R) == 8) {
#pragma unroll
        for (int v = 0; v < S; ++v)
            if (v < NF || v >= Y::ADV) f.in[v] = prim[v];
    }
    if (M == kModesAll && a.rk != kRkNone && a.base_is_in) {
#pragma unroll
        for (int v = 0; v < S; ++v) f.base[v] = f.in[v];
    }
}

// Waves per SIMD the kernel is compiled for.  FP64: two, with 127 to 255
// VGPRs and the next rows' loads a whole pass ahead.  At three (168 VGPRs) the
// contracted x and y march spills 20 bytes, or takes its loads late: 512^3
// 8.24 and 7.69 against 7.35 ms per launch.  On unequal widths, where a lane keeps
// its cell's 27 x coefficients, the x and y march with two fluids spills even so:
// plain 28 bytes of scratch per lane in 2D and 84 in 3D (92 with PO), FP32 bulk
// 16 and 64 at its three waves.
template <typename R>
constexpr int march_waves() { return sizeof(R) == 4 ? 3 : 2; }

// PO: also stores the primitive values of the interior cells (plain form, the
// right-hand side whose caller asks for them; the ghost cells' come from
// k_bc_prim).  A pass of its own read the state for it: 256^3 cells 3.24 ->
// 2.91 ms with it stored here, 1400 x 1300 251 -> 225 us.
template <int NF, int D, int MD, typename R, bool WX, int UNI, bool PO = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(march_waves<R>(), march_waves<R>()))) void k_march(const SweepArgs a) {
    static_assert((MD == 1 && WX) || (!WX && D == 3), "y march with the x faces, y and z march");
    static_assert(sizeof(R) == 8 || !UNI, "FP32 marches are for unequal widths");
    using Y = Sys<NF, D>;
    constexpr int S = Y::S;
    constexpr int PN = 2;
    constexpr int FM = finish_modes<D, WX, R, false>();
    constexpr int W = WX ? kMarchCellsXY : kMarchCellsZ;
    constexpr int HX = WX ? kMarchHaloXY : 0;
    constexpr int HL = WX ? PN : 0;            // ring entries before lane 0's
    constexpr int RW = 64 + 2 * HL;            // entries of a ring row
    constexpr int HB = sizeof(R) == 8 ? 4 : 8; // rows per batch of the entries around the lanes'
    constexpr bool CANON = UNI == kCanonCoef;
    // the RK base: the z march adds the first kBaseOnZFused variables
    constexpr int BLO = MD == 1 && D == 3 ? kBaseOnZFused : 0, BHI = MD == 1 ? S : kBaseOnZFused;
    // whether rhs holds another direction's part: in 3D the sums begin in the
    // z march, or in the plain form in the x and y march or the x sweep
    constexpr bool RHS = D == 3 && (MD == 2 ? FM == kModesAll : WX ? FM != kModesAll : true);
    __shared__ R ring[3][S][RW];
    __shared__ R halo[WX ? S : 1][HB][4];
    // momentum and energy of the ring's rows, this lane's cell
    constexpr bool KEEP = WX && sizeof(R) == 8 && (FM == kModesFoldLast || D == 2);
    constexpr int NK = KEEP ? D + 1 : 0;
    __shared__ double kept[KEEP ? 3 : 1][KEEP ? NK : 1][64];
    double ck[KEEP ? NK : 1], ko[KEEP ? NK : 1]; // of row r and of row r-3

    auto args = [&]() -> const SweepArgs & {
        if constexpr (CANON)
            return a;
        else
            return fresh_args();
    };
    // Blocks: groups of kMarchGroup neighbouring column sets take all chunks
    // before the next group, so the rows two chunks share are still in L2.
    const long bid = xcd_logical_block(blockIdx.x, a.nblocks);
    const long grp = bid / ((long)kMarchGroup * a.nchunk);
    const int rem = (int)(bid - grp * (long)kMarchGroup * a.nchunk);
    const int gw = (int)min((long)kMarchGroup, (long)a.ntile - grp * kMarchGroup);
    const int ch = rem / gw;
    const long set = grp * kMarchGroup + rem % gw;
    const int lane = threadIdx.x;
    const int s = MD == 1 ? a.n : a.p;
    const int r0 = ch * a.chunk, r1 = min(r0 + a.chunk, s + 1); // rows r0 .. r1-1 are finished

    // Entry e (ring entry of lane l: e = l + HL) of the wave is entry G0 + e
    // of the rows of the outer index t set end to end, a.rl entries each, the
    // first HX of them ghost cells.
    const long G0 = set * W - (WX ? 1 : 0) - HL + HX;
    const int t0 = (int)(max(G0, 0L) / a.rl);
    const long gp = MD == 1 ? a.nxg : a.nxg * a.nyg, gt = MD == 1 ? a.nxg * a.nyg : a.nxg;
    const long rp = MD == 1 ? (long)(a.m + 1) : (long)(a.m + 1) * (a.n + 1);
    const long rt = MD == 1 ? (long)(a.m + 1) * (a.n + 1) : (long)(a.m + 1);
    const int touter = MD == 1 ? a.p : a.n;
    const long gb = MD == 1 ? ghost_off(a, -HX, 0, t0) : ghost_off(a, 0, t0, 0);
    const long rb = MD == 1 ? interior_off(a, 0, 0, t0) : interior_off(a, 0, t0, 0);
    // Offsets are 32-bit ones from the variables' first elements (the host
    // checks that a variable is below 4 GiB): the pointers are then used as
    // loaded, with no address arithmetic per access.
    auto entry = [&](int e, int &t, int &xe) { // clamped to the ghosted field
        const long g = max(G0 + e, 0L) - (long)t0 * a.rl;
        const int dt = (int)g / a.rl;
        xe = min((int)g - dt * a.rl, a.m + HX + (WX ? a.b : 0));
        t = t0 + dt;
        if (t > touter) t = touter, xe = a.m + HX;
    };
    int t, xe;
    entry(lane + HL, t, xe);
    const int x = xe - HX; // this lane's cell
    const unsigned own = (unsigned)gb + (unsigned)(t - t0) * (unsigned)gt + (unsigned)xe;
    const unsigned rown = (unsigned)rb + (unsigned)(t - t0) * (unsigned)rt + (unsigned)min(max(x, 0), a.m);
    const bool fin_lane = x >= 0 && x <= a.m && set * W + lane - (WX ? 1 : 0) + HX < (long)a.rl * (touter + 1) &&
                          (!WX || (lane >= 1 && lane <= W));
    // entries 0, 1 and RW-2, RW-1 of row q of a batch on lanes 4q .. 4q+3
    const int hq = (lane >> 2) & (HB - 1), he = (lane & 3) + ((lane & 2) ? RW - 4 : 0);
    int ht, hx;
    entry(he, ht, hx);
    const unsigned hoff = (unsigned)gb + (unsigned)(ht - t0) * (unsigned)gt + (unsigned)hx;
    const int rlast = r1 + PN; // last staged row

    double cv[S];
    auto load_row = [&](int r) {
        const SweepArgs &b = args();
        const Off o{0, own + (unsigned)r * (unsigned)gp};
#pragma unroll
        for (int v = 0; v < S; ++v) cv[v] = el(b.qin.v[v], o);
    };

    const R eps = (R)a.eps;
    const CanonK K;
    R cfx[WX && !UNI ? kNCoef : 1];
    if constexpr (WX && !UNI) load_coef<R, 5, false>(a, min(x, a.m + 1), cfx);
    const double ix = WX ? a.inv_ds[min(max(x, 0), a.m)] : 0.0;

    R vrp[S];     // upper-face values of the row before the stencil's centre
    R fl[S], usl; // flux and contact velocity of that row's lower face
    R w0[S];      // row r-4 of this lane's column
#pragma unroll
    for (int v = 0; v < S; ++v) vrp[v] = fl[v] = w0[v] = R(0);
    usl = R(0);
    int sa = 0, sb = 1, sc = 2; // ring slots of rows r-3, r-2, r-1

    const int rs = r0 - 1 - PN; // first staged row
    load_row(rs);
#pragma unroll 1
    for (int r = rs; r <= rlast; ++r) {
        const int q = r - rs;
        if constexpr (WX) {
            if ((q & (HB - 1)) == 0) {
                double hv[S], hp[S];
                const SweepArgs &b = args();
                const Off o{0, hoff + (unsigned)min(r + hq, rlast) * (unsigned)gp};
#pragma unroll
                for (int v = 0; v < S; ++v) hv[v] = el(b.qin.v[v], o);
                cons_to_prim<NF, D>(hv, hp, a.eos);
                if (lane < 4 * HB) {
#pragma unroll
                    for (int v = 0; v < S; ++v) halo[v][hq][lane & 3] = (R)hp[v];
                }
            }
        }
        R pr[S];
        {
            double p[S];
            cons_to_prim<NF, D>(cv, p, a.eos);
#pragma unroll
            for (int v = 0; v < S; ++v) pr[v] = (R)p[v];
#pragma unroll
            for (int v = 0; v < NK; ++v) ck[v] = cv[Y::MOM + v];
            if constexpr (PO) {
                if (r >= r0 && r < r1 && fin_lane) {
                    const SweepArgs &b = args();
                    const Off o{0, own + (unsigned)r * (unsigned)gp};
#pragma unroll
                    for (int v = 0; v < S; ++v) el(b.prim.v[v], o) = p[v];
                }
            }
        }
        load_row(min(r + 1, rlast));
        // Row r into the ring over row r-3, whose own entries stay in w0.
        auto turn = [&]() {
            R(*ra)[RW] = ring[sa];
            wave_lds_sync();
#pragma unroll
            for (int v = 0; v < S; ++v) {
                w0[v] = ra[v][lane + HL];
                ra[v][lane + HL] = pr[v];
            }
#pragma unroll
            for (int v = 0; v < NK; ++v) {
                ko[v] = kept[sa][v][lane];
                kept[sa][v][lane] = ck[v];
            }
            if constexpr (WX) {
                if (lane < 4) {
#pragma unroll
                    for (int v = 0; v < S; ++v) ra[v][he] = halo[v][q & (HB - 1)][lane];
                }
            }
            wave_lds_sync();
        };
        bool turned = false;
        const int jc = r - PN, jr = jc - 1; // centre of the stencil; row to finish
        R(*ra)[RW] = ring[sa];
        if (jc >= r0 - 1) {
            FinishIn<S> fin;
            const int jl = max(jr, r0); // (its operands are loaded in the passes before the first finish too)
            const Off go{0, own + (unsigned)jl * (unsigned)gp}, ro{0, rown + (unsigned)jl * (unsigned)rp};
            const bool finish = jr >= r0 && fin_lane;
            march_load_acc<NF, D, RHS, FM>(args(), fresh_args(), go, ro, BLO, BHI, fin);
            if constexpr (!WX) {
                march_load_in<NF, D, R, WX, FM>(args(), go, fin);
            }
            // 1. marching direction: both faces of cell jc, then its lower face
            R f[S], us;
            {
                const SweepArgs &b = args();
                R qL[S], qR[S], cf[kNCoef];
                if constexpr (!CANON) {
                    if constexpr (UNI) {
#pragma unroll
                        for (int c = 0; c < kNCoef; ++c)
                            cf[c] = WX ? b.ucf2[c] : b.ucf[c];
                    } else {
                        const double *tab = WX ? b.coef2 : b.coef;
                        const long nc = WX ? b.ncell2 : b.ncell;
#pragma unroll
                        for (int c = 0; c < kNCoef; ++c) cf[c] = (R)uniform_load(tab, (long)c * nc + (jc + b.b));
                    }
                }
                const R(*rb_)[RW] = ring[sb], (*rc_)[RW] = ring[sc];
                // (the next variable's entries are read before this one's
                // arithmetic, here and below: with two waves per SIMD the
                // LDS latency shows)
                R nx[3] = {ra[0][lane + HL], rb_[0][lane + HL], rc_[0][lane + HL]};
#pragma unroll
                for (int v = 0; v < S; ++v) {
                    const R st[5] = {w0[v], nx[0], nx[1], nx[2], pr[v]};
                    if (v + 1 < S) {
                        nx[0] = ra[v + 1][lane + HL];
                        nx[1] = rb_[v + 1][lane + HL];
                        nx[2] = rc_[v + 1][lane + HL];
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    R vr;
                    weno_both<5, R, UNI>(st, cf, eps, qR[v], vr, K);
                    qL[v] = vrp[v];
                    vrp[v] = vr;
                }
                hold(vrp);
                hold(qR);
                const int mb = WX ? b.bc2_beg : b.bc_beg, me = WX ? b.bc2_end : b.bc_end;
                if (jc == 0 && mb == -4) {
#pragma unroll
                    for (int v = 0; v < S; ++v) qL[v] = qR[v];
                }
                if (jc == s + 1 && me == -4) {
#pragma unroll
                    for (int v = 0; v < S; ++v) qR[v] = qL[v];
                }
                hllc_face<NF, D, MD, R>(qL, qR, b.eos, f, us);
                hold(f);
            }
            if (jr >= r0) {
                if constexpr (!WX) {
                    if (finish) {
                        R pv[S];
#pragma unroll
                        for (int v = 0; v < S; ++v) pv[v] = ra[v][lane + HL];
                        march_prim_in<NF, D, R, FM>(args(), pv, fin);
                    }
                    if (finish)
                        finish_cell<NF, D, R, FM, false>(args(), go, ro, a.inv_ds[jr], fl, f, usl, us, fin, BLO, BHI, x, t);
                } else {
                    // 2. x faces of row jr
                    const double iy = a.inv_ds2[jr];
                    double acc[S];
                    {
                        double dfy[S];
#pragma unroll
                        for (int v = 0; v < S; ++v) dfy[v] = to_d(fl[v]) - to_d(f[v]);
                        const double sy = args().fold ? args().cdt * iy : iy;
#pragma unroll
                        for (int v = 0; v < S; ++v)
                            acc[v] = finish_y_part<R>(
                                args(), args().fold, sy, dfy[v], v >= BLO && v < BHI, [&] { return fin.rhs[v]; },
                                [&] { return fin.base[v]; });
                        hold(acc);
                    }
                    const double duy = to_d(us) - to_d(usl);
                    R fx[S], usx;
                    {
                        const SweepArgs &b = args();
                        R qL[S], qR[S], cf[kNCoef];
                        if constexpr (!CANON && UNI) {
#pragma unroll
                            for (int c = 0; c < kNCoef; ++c) cf[c] = b.ucf[c];
                        }
                        R nx[5];
#pragma unroll
                        for (int w = 0; w < 5; ++w) nx[w] = ra[0][lane + w];
#pragma unroll
                        for (int v = 0; v < S; ++v) {
                            R st[5], vl;
#pragma unroll
                            for (int w = 0; w < 5; ++w) st[w] = nx[w];
                            if (v + 1 < S) {
#pragma unroll
                                for (int w = 0; w < 5; ++w) nx[w] = ra[v + 1][lane + w];
                                __builtin_amdgcn_sched_barrier(0);
                            }
                            weno_both<5, R, UNI>(st, UNI ? cf : cfx, eps, vl, qL[v], K);
                            qR[v] = __shfl_down(vl, 1u, 64);
                        }
                        hold(qL);
                        hold(qR);
                        turn();
                        turned = true;
                        march_load_in<NF, D, R, WX, FM>(args(), go, fin);
                        if (x == -1 && b.bc_beg == -4) {
#pragma unroll
                            for (int v = 0; v < S; ++v) qL[v] = qR[v];
                        }
                        if (x == b.m && b.bc_end == -4) {
#pragma unroll
                            for (int v = 0; v < S; ++v) qR[v] = qL[v];
                        }
                        hllc_face<NF, D, 0, R>(qL, qR, b.eos, fx, usx);
                    }
                    double dfx[S];
#pragma unroll
                    for (int v = 0; v < S; ++v) dfx[v] = to_d(__shfl_up(fx[v], 1u, 64)) - to_d(fx[v]);
                    const double dux = to_d(usx) - to_d(__shfl_up(usx, 1u, 64));
#pragma unroll
                    for (int v = 0; v < NK; ++v) fin.in[Y::MOM + v] = ko[v];
                    if (finish) march_prim_in<NF, D, R, FM>(args(), w0, fin);
                    if (finish)
                        finish_xy<NF, D, R, false>(args(), fresh_args(), go, ro, ix, iy, dfx, dux, duy, fin, x, jr,
                                            [&](int v, bool, double) { return acc[v]; });
                }
            }
#pragma unroll
            for (int v = 0; v < S; ++v) fl[v] = f[v];
            usl = us;
        }
        if (!turned) turn();
        const int so = sa;
        sa = sb, sb = sc, sc = so;
    }
}

} // inline namespace MFC_FORM
} // namespace mfc
