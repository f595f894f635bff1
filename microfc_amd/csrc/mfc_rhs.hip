// mfc_rhs.hip -- C ABI of the MI355X RHS library (declared in include/mfc_rhs.h)
// plus the small kernels around the sweeps: ghost-cell fill, cons->prim,
// the CFL max-reduction and the pointwise RK update.
#include "mfc_launch.hpp"
#include "mfc_viscous.hpp"

#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

extern "C" {
#include "../../include/mfc_rhs.h"
}

namespace mfc {
const MlpFrags *mlp_frags();
#define MFC_DECLARE_SWEEP(NF, FORM) \
    template <> int launch_sweep<NF, FORM>(const SweepLaunch &, const SweepArgs &, hipStream_t);
#define MFC_DECLARE_SWEEPS(FORM) \
    MFC_DECLARE_SWEEP(1, FORM) MFC_DECLARE_SWEEP(2, FORM) MFC_DECLARE_SWEEP(3, FORM) MFC_DECLARE_SWEEP(4, FORM)
#define MFC_DECLARE_SWEEPS_WIDE(FORM)                                                                 \
    MFC_DECLARE_SWEEPS(FORM) MFC_DECLARE_SWEEP(5, FORM) MFC_DECLARE_SWEEP(6, FORM) MFC_DECLARE_SWEEP(7, FORM) \
    MFC_DECLARE_SWEEP(8, FORM) MFC_DECLARE_SWEEP(9, FORM) MFC_DECLARE_SWEEP(10, FORM)
MFC_DECLARE_SWEEPS_WIDE(kFormF64)
MFC_DECLARE_SWEEPS(kFormF32)
MFC_DECLARE_SWEEPS_WIDE(kFormF64Fast)
#undef MFC_DECLARE_SWEEPS_WIDE
#undef MFC_DECLARE_SWEEPS
#undef MFC_DECLARE_SWEEP
} // namespace mfc

using namespace mfc;

constexpr int kReduceBlocks = 8192; // the stability pass: 32 blocks of 256 threads per CU
constexpr int kMaxDevices = 64;
// No result of the CFL reduction: a signalling NaN, which no arithmetic returns.
constexpr uint64_t kPending = 0x7FF4A5A5A5A5A5A5ull;
constexpr long kPolls = 100000;

// Block partials of the allocation-free CFL reduction (mfc_cfl_dt_noalloc):
// one copy of this array per GPU, 64 KiB, held until the process ends.  In
// host code its name is not a device address; kernels get the address that
// hipGetSymbolAddress returned for the current device (g_scratch_dev).
static __device__ __align__(256) double scratch[kReduceBlocks];
// Blocks of the running CFL reduction that are done (k_icfl, which leaves it 0).
static __device__ unsigned icfl_done;

namespace {

// Held by the entry points that reduce over the cells, each until its value is
// on the host: they share one block counter per GPU and one result word
// (k_icfl), and all but mfc_cfl_dt_noalloc the case's array of partials.
std::mutex g_reduce;
// The result word, pinned; made by the first mfc_rhs_init and held, as the
// counter and `scratch` are, until the process ends (made per case, an init took
// 244 instead of 202 us).
double *g_result = nullptr;

// Device addresses of `scratch` and `icfl_done` on each GPU, looked up once per
// device by mfc_rhs_init with that device current.
double *g_scratch_dev[kMaxDevices] = {};
unsigned *g_done_dev[kMaxDevices] = {};

constexpr int kNumFluidsBuilt = 10;   // the FP64 forms (every num_fluids the reference allows)
constexpr int kNumFluidsBuiltF32 = 4; // the FP32-bulk and learned forms
// Variables of the RK base that the z sweep of a contracted 3D RK stage
// adds (the y sweep adds the rest).  The step moves the same bytes for any
// split (512^3: 50.6-50.7 ms per step with 0, 2, 3 or 4); half on each
// balances the two sweeps (launches of 5.5 and 5.8 ms instead of 5.0 and
// 6.3 with the whole base on y).
constexpr int kBaseOnZ = 4;
// A grid direction counts as uniform in the contracted and FP32 forms when
// every cell's WENO coefficients are within this relative distance of the
// first reconstructed cell's.  Equal widths on paper differ by the rounding
// of the cell boundaries: 768 cells on [0, 1] give coefficients 2.6e-13
// apart, which moves the RHS by about as much relative to its scale, well
// inside the contracted form's 1e-12.  The plain FP64 form keeps the
// per-cell coefficients unless they are equal bit for bit.
constexpr double kUniformRelTol = 5e-13;
// WENO5 coefficients of cells of equal width (plane order of mfc_device.hpp):
// what the contracted form runs with where every cell lies within
// kUniformRelTol of them too.
constexpr double kCanon[kNCoef] = {
    1.0 / 3, -5.0 / 6, -1.0 / 6, -1.0 / 3, -2.0 / 3, 1.0 / 6, -1.0 / 6, 2.0 / 3,   1.0 / 3,
    1.0 / 6, 5.0 / 6,  -1.0 / 3, 0.1,      0.6,      0.3,     0.3,      0.6,       0.1,
    4.0 / 3, -11.0 / 3, 10.0 / 3, 4.0 / 3, -5.0 / 3, 4.0 / 3, 10.0 / 3, -11.0 / 3, 4.0 / 3};
constexpr bool kFuseXY = true;
// Waves of a march in FP64 and in FP32 (march_waves), or of k_rows_x, that the
// chip runs at a time; the fewest rows of a grid that marches, and of a chunk.
constexpr int kMarchSlots = 8 * 256, kMarchSlots32 = 12 * 256, kMarchRowsMin = 16, kMarchChunkMin = 8;
// The time of `waves` of a march on so many slots, in times of one: one round
// as long as all have a place at once, else the last round is half empty.  With
// that half round added throughout and 16 rows the least of a chunk, a few waves
// were left for a second round: FP32 bulk on unequal widths 115^3 904 -> 722,
// 120^3 1005 -> 804 us per step (800 and 909 in the separate sweeps), plain 4096
// x 2048 2725 -> 2596 (2605 in the tiles).
double chunk_rounds(double waves, int slots) {
    const double r = waves / slots;
    return r <= 1.0 ? 1.0 : r + 0.5;
}
// Cells from which a march (k_march) takes over, where both were measured
// (ms per RK3 step, tile kernels -> marches; two fluids):
//  * equal widths, 3D: contracted FP64 128^3 0.82 -> 0.82, 200^3 2.72 -> 2.63,
//    512^3 42.1 -> 36.8; plain FP64 128^3 1.45 -> 1.43; one RHS at 256^3
//    3.52 -> 3.24;
//  * equal widths, 2D: contracted 2048^2 0.73 -> 0.79, 4096^2 2.70 -> 2.54;
//    plain 2048^2 1.36 -> 1.50, 4096^2 5.13 -> 5.02;
//  * other widths, against the separate sweeps: contracted 1024^2 0.326 ->
//    0.331, 1500^2 0.78 -> 0.52, 4096^2 5.53 -> 3.10, 96^3 0.51 -> 0.48, 128^3
//    1.36 -> 0.93, 200^3 4.95 -> 2.97; plain 1024^2 0.49 -> 0.56, 1500^2 1.02 ->
//    0.92, 4096^2 7.41 -> 5.74, 96^3 0.77 -> 0.79, 200^3 6.74 -> 4.93; FP32 bulk
//    1024^2 0.26 -> 0.29, 2048^2 1.22 -> 0.86, 96^3 0.41 -> 0.48, 200^3 4.10 ->
//    3.33.
//  * three fluids, other widths, y and z against the separate sweeps:
//    contracted 150 x 112 x 92 1.38 -> 1.12, 180 x 130 x 90 1.79 -> 1.40; plain
//    150 x 112 x 92 1.86 -> 1.60; FP32 bulk 200^3, z alone 4.93 -> 4.81 (with y
//    4.88); equal widths 256^3, z alone: contracted 8.70 -> 8.26 (with y 8.41),
//    plain 14.3 -> 13.7;
//  * just above these lines, with the chunks of chunk_rounds: equal widths 4096
//    x 2048 contracted 1.67 -> 1.28, plain 2.61 -> 2.54 (one fluid 2.09 -> 2.00);
//    other widths 1300^2 contracted 0.570 -> 0.361, plain 0.755 -> 0.638, FP32
//    bulk 0.478 -> 0.376 (one fluid 0.318 -> 0.293); 120^3 contracted 1.08 ->
//    0.73, plain 1.43 -> 1.18, FP32 bulk 0.909 -> 0.803 (one fluid 0.675 ->
//    0.559).
// The FP32-bulk form on equal widths keeps its tiles (300 x 250 x 200 4.75 ->
// 4.91): with half the LDS and registers they fill the SIMDs already.
constexpr double kMarchUniform2D = 8e6, kMarchUniform3D = 3e6, kMarchPerCell = 1.5e6;

thread_local std::string g_err;

int fail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

#define HIPCHK(expr)                                                                   \
    do {                                                                               \
        hipError_t e_ = (expr);                                                        \
        if (e_ != hipSuccess) return fail(-3, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

struct Dir {
    int s = 0;
    double *coef = nullptr;   // device, 27 x ncell
    double *inv_ds = nullptr; // device, s+1
    double *ds_dev = nullptr; // device, ds(0..s)
    double *cc_dev = nullptr; // device, ghosted cell centres s_cc(-b..s+b)
    double *inv_dsg = nullptr; // device, 1/ds(i) for i = -b..s+b (weno_Re_flux gradients)
    std::vector<double> coef_h, ds_h;
    bool ready = false;
    // every reconstructed cell has the same coefficients: bit for bit in the
    // plain FP64 form, to kUniformRelTol in the others
    bool uniform = false;
    // contracted form, WENO5: uniform, and every reconstructed cell's
    // coefficients within kUniformRelTol of equal widths' (kCanon)
    bool canon = false;
    double ucf[kNCoef] = {};
    bool uniform_wide = false; // the same over every cell the coefficients are set for (-b+polyn..s+b-polyn)
};

struct State {
    bool init = false;
    mfc_params prm{};
    int D = 1, S = 0, b = 0, polyn = 0;
    long nxg = 0, nyg = 0, nzg = 0, ng = 0, nint = 0;
    Dir dir[3];
    hipStream_t own = nullptr, stream = nullptr;
    double *partials = nullptr; // 2 * kReduceBlocks doubles
    double *scratch = nullptr;  // this device's `scratch` array (kReduceBlocks doubles)
    unsigned *count = nullptr;  // this device's `icfl_done`
    double *scratch_state = nullptr; // S*ng doubles, RK3 stage buffer
    bool visc = false;               // any fluid_pp%Re > 0
    ViscParams vp{};
    bool wrf = false;                // viscous with weno_Re_flux: WENO-reconstructed velocity gradients
    double *visc_grad = nullptr;     // D*D planes of ng: cell-centred velocity gradients (weno_Re_flux)
} G;

// ---------------------------------------------------------------------------
// Optional per-kernel timing with HIP events on the library's stream.
enum KernelId { kKBcFill = 0, kKConsToPrim, kKSweepX, kKSweepY, kKSweepZ, kKIcfl, kKRk1, kKViscous, kKSweepXY,
                // which kernel a sweep was, counted beside its direction's id
                kKTileXY, kKMarchXY, kKMarchZ, kKMarchY, kKRowsX, kKStage, kKCount };
const char *const kKernelNames[kKCount] = {"bc_fill", "cons_to_prim", "sweep_x", "sweep_y", "sweep_z", "icfl",
                                           "rk1_update", "viscous", "sweep_xy", "tile_xy", "march_xy", "march_z",
                                           "march_y", "rows_x", "stage"};

struct Timing {
    bool on = false;
    struct Rec {
        int id, sub;
        hipEvent_t a, b;
    };
    std::vector<Rec> pending;
    std::vector<hipEvent_t> pool;
    double total_ms[kKCount] = {};
    long count[kKCount] = {};
    hipEvent_t get() {
        if (!pool.empty()) {
            hipEvent_t e = pool.back();
            pool.pop_back();
            return e;
        }
        hipEvent_t e = nullptr;
        if (hipEventCreate(&e) != hipSuccess) return nullptr;
        return e;
    }
} T;

struct TimedScope {
    int id, sub;
    hipEvent_t a = nullptr;
    explicit TimedScope(int k, int s = -1) : id(k), sub(s) { // k < 0: not timed; s >= 0: counted there too
        if (k >= 0 && T.on && (a = T.get())) (void)hipEventRecord(a, G.stream);
    }
    ~TimedScope() {
        if (!a) return;
        hipEvent_t b = T.get();
        if (!b) return;
        (void)hipEventRecord(b, G.stream);
        T.pending.push_back({id, sub, a, b});
    }
};

int timing_flush() {
    if (T.pending.empty()) return 0;
    HIPCHK(hipStreamSynchronize(G.stream));
    for (auto &r : T.pending) {
        float ms = 0.f;
        HIPCHK(hipEventElapsedTime(&ms, r.a, r.b));
        for (int k : {r.id, r.sub})
            if (k >= 0) {
                T.total_ms[k] += ms;
                T.count[k] += 1;
            }
        T.pool.push_back(r.a);
        T.pool.push_back(r.b);
    }
    T.pending.clear();
    return 0;
}

// ---------------------------------------------------------------------------
// input checks: src/simulation/m_start_up.fpp:117-290 (the parts that apply)
int check_params(const mfc_params &p) {
    if (p.m <= 0) return fail(-1, "Unsupported value of m");
    if (p.n < 0) return fail(-1, "Unsupported value of n");
    if (p.p < 0) return fail(-1, "Unsupported value of p");
    if (p.p > 0 && p.n == 0) return fail(-1, "p > 0 requires n > 0");
    if (p.num_fluids < 1 || p.num_fluids > MFC_NUM_FLUIDS_MAX) return fail(-1, "Unsupported value of num_fluids");
    if (p.num_fluids > kNumFluidsBuilt)
        return fail(-1, "num_fluids = %d: kernels are built for 1..%d fluids", p.num_fluids, kNumFluidsBuilt);
    if (p.weno_order != 1 && p.weno_order != 3 && p.weno_order != 5) return fail(-1, "Unsupported value of weno_order");
    if (p.m + 1 < 5 * p.weno_order) return fail(-1, "Unsupported combination of values of m and weno_order");
    if (p.n > 0 && p.n + 1 < 5 * p.weno_order) return fail(-1, "Unsupported combination of values of n and weno_order");
    if (p.p > 0 && p.p + 1 < 5 * p.weno_order) return fail(-1, "Unsupported combination of values of p and weno_order");
    if (!(p.weno_eps > 0.0) || p.weno_eps > 1e-6) return fail(-1, "Unsupported value of weno_eps");
    if (p.time_stepper < 1 || p.time_stepper > 3) return fail(-1, "Unsupported value of time_stepper");
    const int bcs[3][2] = {{p.bc_x_beg, p.bc_x_end}, {p.bc_y_beg, p.bc_y_end}, {p.bc_z_beg, p.bc_z_end}};
    const char *nm[3] = {"bc_x", "bc_y", "bc_z"};
    const int D = 1 + (p.n > 0) + (p.p > 0);
    for (int d = 0; d < D; ++d) {
        for (int e = 0; e < 2; ++e)
            if (bcs[d][e] < -12 || bcs[d][e] > -1)
                return fail(-1, "Unsupported value of %s%%%s", nm[d], e ? "end" : "beg");
        if ((bcs[d][0] == -1) != (bcs[d][1] == -1))
            return fail(-1, "Unsupported combination of values of %s%%beg and %s%%end", nm[d], nm[d]);
    }
    for (int i = 0; i < p.num_fluids; ++i) {
        if (!(p.gammas[i] > 0.0)) return fail(-1, "Unsupported value of fluid_pp(%d)%%gamma", i + 1);
        if (p.pi_infs[i] < 0.0) return fail(-1, "Unsupported value of fluid_pp(%d)%%pi_inf", i + 1);
    }
    if (p.precision != MFC_PREC_FP64 && p.precision != MFC_PREC_FP32_BULK && p.precision != MFC_PREC_FP32_LEARNED &&
        p.precision != MFC_PREC_FP64_FAST)
        return fail(-1, "Unsupported precision");
    const bool f64 = p.precision == MFC_PREC_FP64 || p.precision == MFC_PREC_FP64_FAST;
    if (!f64 && p.num_fluids > kNumFluidsBuiltF32)
        return fail(-1, "num_fluids = %d: the FP32 forms are built for 1..%d fluids", p.num_fluids,
                    kNumFluidsBuiltF32);
    if (p.precision == MFC_PREC_FP32_LEARNED && p.weno_order != 5)
        return fail(-1, "learned WENO weights need weno_order = 5");
    bool visc = false;
    for (int i = 0; i < p.num_fluids; ++i)
        for (int r = 0; r < 2; ++r) visc = visc || p.Re[i][r] > 0.0;
    if (visc && D > 2) return fail(-1, "viscous terms are 1D and 2D only, as in the reference");
    if (visc && p.precision != MFC_PREC_FP64) return fail(-1, "viscous terms run in the plain FP64 form only");
    if (visc && p.num_fluids > kViscFluidsMax)
        return fail(-1, "viscous kernels are built for 1..%d fluids", kViscFluidsMax);
    // The FP64 weight divisions (ndiv) equal IEEE division while the squared
    // smoothness indicators stay within [1e-200, 1e100], which weno_eps >=
    // 1e-100 guarantees from below.
    if (f64 && p.weno_order > 1 && !(p.weno_eps >= 1e-100))
        return fail(-1, "weno_eps below 1e-100 is not supported in FP64 (the weight division is exact for "
                        "weno_eps >= 1e-100)");
    // The contracted form scales the WENO5 weights by the product of the
    // three squared smoothness indicators and normalises both faces of a
    // cell with one reciprocal of the product of their weight sums (>=
    // weno_eps^8 / 100): normal for weno_eps >= 1e-25, finite while the
    // stencil differences stay below about 1e18.
    if (p.precision == MFC_PREC_FP64_FAST && p.weno_order > 1 && !(p.weno_eps >= 1e-25))
        return fail(-1, "weno_eps below 1e-25 is not supported in the contracted FP64 form (the scaled weights "
                        "and the product of a cell's two weight sums must stay normal)");
    // In FP32, beta^2 >= weno_eps^2 must stay a normal float and d/beta^2 finite.
    if (!f64 && p.weno_order > 1 && !(p.weno_eps >= 1e-18))
        return fail(-1, "weno_eps below 1e-18 is not supported in the FP32 forms (its square underflows)");
    return 0;
}

// ---------------------------------------------------------------------------
// WENO coefficient tables on the host: src/simulation/m_weno.fpp:168-363.
// Same plane layout as mfc_device.hpp; x**2d0 is evaluated as x*x.
inline double sq(double x) { return x * x; }

void weno_tables(int s, int b, int order, const double *cb0, std::vector<double> &out) {
    const long nc = s + 2 * b + 1;
    const double *cb = cb0 + 1 + b; // cb[i] = s_cb(i)
    const int polyn = (order - 1) / 2;
    out.assign(27 * nc, 0.0);
    if (order == 1) return;
    auto C = [&](int plane, int j) -> double & { return out[(long)plane * nc + j + b]; };
    for (int i = -b - 1 + polyn; i <= s + b - 1 - polyn; ++i) {
        const int j = i + 1;
        const double S0 = cb[i], S1 = cb[i + 1], S2 = cb[i + 2], Sm1 = cb[i - 1];
        if (order == 3) {
            C(kCbR + 0, j) = (S0 - S1) / (S0 - S2);
            C(kCbR + 2, j) = (S0 - S1) / (Sm1 - S1);
            C(kCbL + 0, j) = -C(kCbR + 0, j);
            C(kCbL + 2, j) = -C(kCbR + 2, j);
            C(kDR + 0, j) = (Sm1 - S1) / (Sm1 - S2);
            C(kDL + 0, j) = (Sm1 - S0) / (Sm1 - S2);
            C(kDR + 1, j) = 1.0 - C(kDR + 0, j);
            C(kDL + 1, j) = 1.0 - C(kDL + 0, j);
            C(kBeta + 0, j) = 4.0 * sq(S0 - S1) / sq(S0 - S2);
            C(kBeta + 3, j) = 4.0 * sq(S0 - S1) / sq(Sm1 - S1);
            continue;
        }
        const double S3 = cb[i + 3], Sm2 = cb[i - 2];
        const double h4 = 4.0 * sq(S0 - S1);
        C(kCbR + 0, j) = ((S0 - S1) * (S1 - S2)) / ((S0 - S3) * (S3 - S1));
        C(kCbR + 2, j) = ((Sm1 - S1) * (S1 - S0)) / ((Sm1 - S2) * (S2 - S0));
        C(kCbR + 3, j) = ((S0 - S1) * (S1 - S2)) / ((Sm1 - S1) * (Sm1 - S2));
        C(kCbR + 5, j) = ((S0 - S1) * (S1 - Sm1)) / ((Sm2 - S0) * (Sm2 - S1));
        C(kCbL + 0, j) = ((S1 - S0) * (S0 - S2)) / ((S0 - S3) * (S3 - S1));
        C(kCbL + 2, j) = ((S0 - Sm1) * (S0 - S1)) / ((Sm1 - S2) * (S0 - S2));
        C(kCbL + 3, j) = ((S1 - S0) * (S0 - S2)) / ((Sm1 - S1) * (Sm1 - S2));
        C(kCbL + 5, j) = ((Sm1 - S0) * (S0 - S1)) / ((Sm2 - S0) * (Sm2 - S1));
        C(kCbR + 1, j) = ((S0 - S2) + (S1 - S3)) / ((S0 - S2) * (S0 - S3)) * ((S0 - S1));
        C(kCbR + 4, j) = ((Sm2 - S1) + (Sm1 - S1)) / ((Sm1 - S1) * (S1 - Sm2)) * ((S1 - S0));
        C(kCbL + 1, j) = ((S0 - S2) + (S0 - S3)) / ((S0 - S2) * (S0 - S3)) * ((S1 - S0));
        C(kCbL + 4, j) = ((Sm2 - S0) + (Sm1 - S1)) / ((Sm2 - S1) * (S1 - Sm1)) * ((S0 - S1));
        C(kDR + 0, j) = ((Sm2 - S1) * (S1 - Sm1)) / ((Sm2 - S3) * (S3 - Sm1));
        C(kDR + 2, j) = ((S1 - S2) * (S1 - S3)) / ((Sm2 - S2) * (Sm2 - S3));
        C(kDL + 0, j) = ((Sm2 - S0) * (S0 - Sm1)) / ((Sm2 - S3) * (S3 - Sm1));
        C(kDL + 2, j) = ((S0 - S2) * (S0 - S3)) / ((Sm2 - S2) * (Sm2 - S3));
        C(kDR + 1, j) = 1.0 - C(kDR + 0, j) - C(kDR + 2, j);
        C(kDL + 1, j) = 1.0 - C(kDL + 0, j) - C(kDL + 2, j);
        const double a10 = S1 - S0, a21 = S2 - S1, a20 = S2 - S0, a31 = S3 - S1, a0m = S0 - Sm1;
        C(kBeta + 0, j) = h4 * (10.0 * sq(a10) + a10 * a21 + sq(a21)) / (sq(S0 - S3) * sq(S1 - S3));
        C(kBeta + 1, j) = h4 * (19.0 * sq(a10) - a10 * a31 + 2.0 * a20 * (a20 + a31)) /
                          ((S0 - S2) * sq(S0 - S3) * a31);
        C(kBeta + 2, j) = h4 * (10.0 * sq(a10) + a10 * (a20 + a31) + sq(a20 + a31)) / (sq(S0 - S2) * sq(S0 - S3));
        C(kBeta + 3, j) = h4 * (10.0 * sq(a10) + sq(a0m) + a0m * a10) / (sq(Sm1 - S2) * sq(S0 - S2));
        C(kBeta + 4, j) = h4 * ((S0 - S1) * (a0m + 20.0 * a10) + (2.0 * a0m + a10) * a20) /
                          ((S1 - Sm1) * sq(Sm1 - S2) * a20);
        C(kBeta + 5, j) = h4 * (10.0 * sq(a10) + a10 * a21 + sq(a21)) / (sq(Sm1 - S1) * sq(Sm1 - S2));
        const double c2m = (S0 - Sm2) + (S0 - Sm1);
        C(kBeta + 6, j) = h4 * (12.0 * sq(a10) + sq(c2m) + 3.0 * c2m * a10) / (sq(Sm2 - S1) * sq(Sm1 - S1));
        C(kBeta + 7, j) = h4 * (19.0 * sq(a10) + ((S0 - Sm2) * (S0 - S1)) + 2.0 * (S1 - Sm1) * ((S0 - Sm2) + (S1 - Sm1))) /
                          ((Sm2 - S0) * sq(Sm2 - S1) * (S1 - Sm1));
        C(kBeta + 8, j) = h4 * (10.0 * sq(a10) + sq(a0m) + a0m * a10) / (sq(Sm2 - S0) * sq(Sm2 - S1));
    }
}

// ---------------------------------------------------------------------------
// small kernels

struct Box {
    int m, n, p, b, bj, bk;
    long nxg, nyg;
};

__device__ __forceinline__ long box_off(const Box &x, int i, int j, int k) {
    return (long)(i + x.b) + x.nxg * ((long)(j + x.bj) + x.nyg * (long)(k + x.bk));
}

// Ghost fill.  The reference fills x ghosts for interior rows, then y ghosts
// over all x, then z ghosts over all x and y, so a corner holds the interior
// cell reached by applying each direction's map in turn, with the momentum
// component normal to each reflecting boundary negated.  Each thread here
// fills one ghost cell with that composed map.  blockIdx.y selects the slab:
// 0: x ghosts (all j, k), 1: y ghosts (interior i, all k), 2: z ghosts
// (interior i, j); together they cover every ghost cell once.
//
// Latency bound on small grids (a few thousand ghost cells): every variable's
// load is issued before the first store (one variable after another, each
// round trip waits for the one before), and the cell's indices come from
// 32-bit divisions.  200 x 150 cells, 7 variables 4.7 -> 3.7 us, 1000 cells 3.3 -> 2.8 us.
constexpr int kBcVars = 8; // variables per round trip
struct BcCodes {
    int xb, xe, yb, ye, zb, ze;
};
// Ghost cell t of slab `slab`: its offset, its source's and the mirrored
// directions; false past the slab's end.
__device__ __forceinline__ bool bc_cell(const Box &x, const BcCodes &bc, int slab, unsigned t, unsigned n0, unsigned n1,
                                        unsigned n2, long &dst, long &src, bool &fx, bool &fy, bool &fz) {
    int i, j, k;
    const unsigned gx = 2 * x.b, gy = 2 * x.bj;
    const unsigned NY = x.n + 1 + gy, NX = x.m + 1;
    if (slab == 0) {
        if (t >= n0) return false;
        const unsigned r = t / gx, gi = t - r * gx, kk = r / NY, jj = r - kk * NY;
        i = (int)gi < x.b ? (int)gi - x.b : x.m + 1 + ((int)gi - x.b);
        j = (int)jj - x.bj;
        k = (int)kk - x.bk;
    } else if (slab == 1) {
        if (t >= n1) return false;
        const unsigned r = t / NX, ii = t - r * NX, kk = r / gy, gj = r - kk * gy;
        i = (int)ii;
        j = (int)gj < x.bj ? (int)gj - x.bj : x.n + 1 + ((int)gj - x.bj);
        k = (int)kk - x.bk;
    } else {
        if (t >= n2) return false;
        const unsigned r = t / NX, ii = t - r * NX, NI = x.n + 1, gk = r / NI, jj = r - gk * NI;
        i = (int)ii;
        j = (int)jj;
        k = (int)gk < x.bk ? (int)gk - x.bk : x.p + 1 + ((int)gk - x.bk);
    }
    fx = fy = fz = false;
    const int si = bc_source(bc.xb, bc.xe, x.m, i, fx);
    const int sj = x.bj ? bc_source(bc.yb, bc.ye, x.n, j, fy) : j;
    const int sk = x.bk ? bc_source(bc.zb, bc.ze, x.p, k, fz) : k;
    dst = box_off(x, i, j, k);
    src = box_off(x, si, sj, sk);
    return true;
}
__global__ __launch_bounds__(256) void k_bc_fill(Fields q, int S, int momxb, Box x, BcCodes bc, unsigned n0, unsigned n1,
                                                 unsigned n2) {
    long dst, src;
    bool fx, fy, fz;
    if (!bc_cell(x, bc, blockIdx.y, blockIdx.x * 256u + threadIdx.x, n0, n1, n2, dst, src, fx, fy, fz)) return;
    for (int v0 = 0; v0 < S; v0 += kBcVars) {
        double val[kBcVars];
#pragma unroll
        for (int u = 0; u < kBcVars; ++u)
            if (v0 + u < S) val[u] = q.v[v0 + u][src];
#pragma unroll
        for (int u = 0; u < kBcVars; ++u) {
            const int v = v0 + u;
            if (v >= S) break;
            const bool neg = (fx && v == momxb) || (fy && v == momxb + 1) || (fz && v == momxb + 2);
            q.v[v][dst] = neg ? -val[u] : val[u];
        }
    }
}

// The ghost fill and the ghost cells' primitive values.
template <int NF, int D>
__global__ __launch_bounds__(256) void k_bc_prim(Fields q, Fields qp, Eos eos, Box x, BcCodes bc, unsigned n0,
                                                 unsigned n1, unsigned n2) {
    using Y = Sys<NF, D>;
    constexpr int S = Y::S;
    long dst, src;
    bool f[3];
    if (!bc_cell(x, bc, blockIdx.y, blockIdx.x * 256u + threadIdx.x, n0, n1, n2, dst, src, f[0], f[1], f[2])) return;
    double c[S], p[S];
#pragma unroll
    for (int v = 0; v < S; ++v) c[v] = q.v[v][src];
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (f[d]) c[Y::MOM + d] = -c[Y::MOM + d];
    cons_to_prim<NF, D>(c, p, eos);
#pragma unroll
    for (int v = 0; v < S; ++v) {
        q.v[v][dst] = c[v];
        qp.v[v][dst] = p[v];
    }
}

template <int NF, int D>
__global__ void k_cons_to_prim(Fields qc, Fields qp, Eos eos, long ng) {
    constexpr int S = Sys<NF, D>::S;
    const long o = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= ng) return;
    double c[S], p[S];
#pragma unroll
    for (int v = 0; v < S; ++v) c[v] = qc.v[v][o];
    cons_to_prim<NF, D>(c, p, eos);
#pragma unroll
    for (int v = 0; v < S; ++v) qp.v[v][o] = p[v];
}

// NaN-propagating maximum: once a NaN is seen it stays.
__device__ __forceinline__ double max_nan(double a, double b) {
    return (a != a || b != b) ? (a != a ? a : b) : (a > b ? a : b);
}

__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = max_nan(v, __shfl_xor(v, off, 64));
    return v;
}

// ICFL of one cell (m_data_output.fpp:197-244) from its S values: primitive
// ones, or conservative ones converted first (FROM_CONS; the values are
// identical because the reference's q_prim_vf is that same conversion).
template <int NF, int D, bool FROM_CONS>
__device__ __forceinline__ double icfl_cell(const double *cv, const Eos &eos, const double *dx, const double *dy,
                                            const double *dz, int i, int j, int k, double dt) {
    using Y = Sys<NF, D>;
    constexpr int S = Y::S;
    double pr[S];
    if constexpr (FROM_CONS) {
        cons_to_prim<NF, D>(cv, pr, eos);
    } else {
#pragma unroll
        for (int v = 0; v < S; ++v) pr[v] = cv[v];
    }
    double rho = 0.0, gam = 0.0, pinf = 0.0;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        rho = rho + pr[f];
        gam = gam + pr[Y::ADV + f] * eos.gammas[f];
        pinf = pinf + pr[Y::ADV + f] * eos.pi_infs[f];
    }
    const double pres = pr[Y::E];
    const double c = sqrt(((gam + 1.0) * pres + pinf) / (gam * rho));
    if constexpr (D == 1) {
        return (dt / dx[i]) * (fabs(pr[Y::MOM]) + c);
    } else if constexpr (D == 2) {
        return dt / min_ref(dx[i] / (fabs(pr[Y::MOM]) + c), dy[j] / (fabs(pr[Y::MOM + 1]) + c));
    } else {
        return dt / min_ref(min_ref(dx[i] / (fabs(pr[Y::MOM]) + c), dy[j] / (fabs(pr[Y::MOM + 1]) + c)),
                            dz[k] / (fabs(pr[Y::MOM + 2]) + c));
    }
}

// Maximum over a block of T threads, valid on its first wave.
template <int T> __device__ __forceinline__ double block_max(double mx) {
    __shared__ double red[T / 64];
    mx = wave_max(mx);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    const double v = wave_max(red[threadIdx.x & (T / 64 - 1)]);
    __syncthreads(); // red may be written again
    return v;
}

// Maximum ICFL over the interior to *result: a block max-reduction by
// wavefront shuffles into partials[blockIdx.x], and the block that finishes
// last reduces the partials (count wraps to 0 with it, ready for the next
// call).  A block takes chunks of kCflChunk consecutive interior cells (x
// fastest), two per thread with both cells' loads issued before either is
// converted.  Two blocks per compute unit on small grids, since the counter
// takes 10 ns a block (the call with 768^2 cells in 1152 blocks of 256 threads
// took 37 us, in 512 of 512 30 us; 1500^2 cells 48.7 us in 2048 blocks, 38.3
// in 512), and up to eight on large ones, where a block takes eight chunks and
// more (320^3 cells 407 us in 512 blocks, 391 in 2048).
// result is pinned host memory.  With the partials reduced by a kernel of
// their own and the value copied to pageable memory, the call took 34 instead
// of 24 us (200^2 cells), 38 instead of 30 us (768^2), 210 instead of 197 us
// (4096^2); then the host stopped waiting for the stream (icfl_reduce).
constexpr int kCflThreads = 512, kCflChunk = 2 * kCflThreads, kCflBlocks = 2048;
// Blocks for so many chunks.
int cfl_blocks(long chunks) {
    return (int)std::min<long>(kCflBlocks, std::max(std::min(chunks, 512L), chunks / 8));
}
template <int NF, int D, bool FROM_CONS>
__global__ __launch_bounds__(kCflThreads) void k_icfl(Fields q, Eos eos, Box x, const double *dx, const double *dy,
                                              const double *dz, double dt, long nint, double *partials,
                                              unsigned *count, double *result) {
    constexpr int S = Sys<NF, D>::S;
    const unsigned nx = x.m + 1, ny = x.n + 1;
    const bool small = nint < (1L << 31); // 32-bit index divisions
    double mx = -INFINITY;
    for (long c0 = (long)blockIdx.x * kCflChunk; c0 < nint; c0 += (long)gridDim.x * kCflChunk) {
        double cv[2][S];
        int ci[2], cj[2], ck[2];
        bool ok[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const long e = c0 + threadIdx.x + kCflThreads * h;
            ok[h] = e < nint;
            const long ee = ok[h] ? e : 0;
            long r;
            if (small) {
                r = (unsigned)ee / nx;
                ck[h] = (int)((unsigned)r / ny);
            } else {
                r = ee / nx;
                ck[h] = (int)(r / ny);
            }
            ci[h] = (int)(ee - r * nx);
            cj[h] = (int)(r - (long)ck[h] * ny);
            const long o = box_off(x, ci[h], cj[h], ck[h]);
#pragma unroll
            for (int v = 0; v < S; ++v) cv[h][v] = q.v[v][o];
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (ok[h]) mx = max_nan(mx, icfl_cell<NF, D, FROM_CONS>(cv[h], eos, dx, dy, dz, ci[h], cj[h], ck[h], dt));
    }
    __shared__ bool last;
    mx = block_max<kCflThreads>(mx);
    if (threadIdx.x == 0) {
        // an exchange that has returned is visible to every block: with a
        // store and a __threadfence (a write-back of L2 per block) instead,
        // 768^2 cells took 50 us
        double old = __hip_atomic_exchange(&partials[blockIdx.x], mx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(old) : : "memory");
        last = atomicInc(count, gridDim.x - 1) == gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    mx = -INFINITY;
    for (unsigned t = threadIdx.x; t < gridDim.x; t += kCflThreads)
        mx = max_nan(mx, __hip_atomic_load(&partials[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    mx = block_max<kCflThreads>(mx);
    if (threadIdx.x == 0) __hip_atomic_store(result, mx, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Stability criteria of one cell (m_data_output.fpp:214-263) from its
// primitive values, for viscous cases: the mixture Reynolds numbers of
// s_convert_species_to_mixture_variables_acc (m_variables_conversion.fpp:
// 210-223), VCFL = maxval(dt/Re)/min(dx, dy)**2 and
// Rc = min(dx(|u|+c), dy(|v|+c))/maxval(1/Re) (1D: dx alone).
template <int NF, int D>
__device__ __forceinline__ void visc_criteria(const double *pr, const Eos &eos, const ViscParams &vp, double dxi,
                                              double dyj, double dt, double &vcfl, double &rc) {
    using Y = Sys<NF, D>;
    double rho = 0.0, gam = 0.0, pinf = 0.0, Re[2];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        rho = rho + pr[f];
        gam = gam + pr[Y::ADV + f] * eos.gammas[f];
        pinf = pinf + pr[Y::ADV + f] * eos.pi_infs[f];
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        double v = -1e6; // dflt_real
        if (vp.size[r] > 0) v = 0.0;
        for (int q = 0; q < vp.size[r]; ++q) v = pr[Y::ADV + vp.idx[r][q]] / vp.res[r][q] + v;
        Re[r] = 1.0 / max_ref(v, 1e-16);
    }
    const double c = sqrt(((gam + 1.0) * pr[Y::E] + pinf) / (gam * rho));
    const double dtre = max_ref(dt / Re[0], dt / Re[1]);
    const double inv = max_ref(1.0 / Re[0], 1.0 / Re[1]);
    if constexpr (D == 1) {
        vcfl = dtre / (dxi * dxi);
        rc = dxi * (fabs(pr[Y::MOM]) + c) / inv;
    } else {
        const double h = min_ref(dxi, dyj);
        vcfl = dtre / (h * h);
        rc = min_ref(dxi * (fabs(pr[Y::MOM]) + c), dyj * (fabs(pr[Y::MOM + 1]) + c)) / inv;
    }
}

// VCFL maximum and Rc minimum over the interior (as the negated maximum of
// -Rc, so both reduce with max_nan); block results to partials[blockIdx.x]
// and partials[gridDim.x + blockIdx.x].
template <int NF, int D>
__global__ __launch_bounds__(256) void k_visc_criteria(Fields q, Eos eos, ViscParams vp, Box x, const double *dx,
                                                       const double *dy, double dt, long nint, double *partials) {
    constexpr int S = Sys<NF, D>::S;
    double mv = -INFINITY, mr = -INFINITY;
    for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < nint; e += (long)gridDim.x * 256) {
        const long r = e / (x.m + 1);
        const int i = (int)(e - r * (x.m + 1));
        const int j = (int)(r % (x.n + 1));
        const long o = box_off(x, i, j, 0);
        double pr[S];
#pragma unroll
        for (int v = 0; v < S; ++v) pr[v] = q.v[v][o];
        double vcfl, rc;
        visc_criteria<NF, D>(pr, eos, vp, dx[i], D > 1 ? dy[j] : 0.0, dt, vcfl, rc);
        mv = max_nan(mv, vcfl);
        mr = max_nan(mr, -rc);
    }
    __shared__ double red[2][4];
    mv = wave_max(mv);
    mr = wave_max(mr);
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = mv;
        red[1][threadIdx.x >> 6] = mr;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = red[0][0], b = red[1][0];
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w) {
            a = max_nan(a, red[0][w]);
            b = max_nan(b, red[1][w]);
        }
        partials[blockIdx.x] = a;
        partials[gridDim.x + blockIdx.x] = b;
    }
}

// Final pass over the block partials: one block of 1024 threads (eight
// partials per thread at 8192 blocks).
__global__ __launch_bounds__(1024) void k_reduce_max(double *partials, int n) {
    double mx = -INFINITY;
    for (int t = threadIdx.x; t < n; t += blockDim.x) mx = max_nan(mx, partials[t]);
    __shared__ double red[16];
    mx = wave_max(mx);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        double v = red[0];
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w) v = max_nan(v, red[w]);
        partials[0] = v;
    }
}

// Pointwise RK1 update q = q + dt*rhs on the interior
// (m_time_steppers.fpp:165-175); in place, so it cannot be fused into a
// stencil sweep that reads q.
__global__ void k_rk1_update(Fields q, Fields rhs, int S, Box x, double dt, long nint) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nint) return;
    const int i = (int)(t % (x.m + 1));
    const long r = t / (x.m + 1);
    const int j = (int)(r % (x.n + 1));
    const int k = (int)(r / (x.n + 1));
    const long o = box_off(x, i, j, k);
    for (int v = 0; v < S; ++v) q.v[v][o] = q.v[v][o] + dt * rhs.v[v][t];
}

// ---------------------------------------------------------------------------
// host helpers

Box box() {
    Box x;
    x.m = G.prm.m;
    x.n = G.prm.n;
    x.p = G.prm.p;
    x.b = G.b;
    x.bj = G.prm.n > 0 ? G.b : 0;
    x.bk = G.prm.p > 0 ? G.b : 0;
    x.nxg = G.nxg;
    x.nyg = G.nyg;
    return x;
}

Eos eos() {
    Eos e;
    for (int i = 0; i < kNumFluidsMax; ++i) {
        e.gammas[i] = G.prm.gammas[i];
        e.pi_infs[i] = G.prm.pi_infs[i];
    }
    return e;
}

int fields(double *const *ptrs, Fields &f, const char *what) {
    if (!ptrs) return fail(-1, "%s: NULL field array", what);
    for (int v = 0; v < kMaxSys; ++v) f.v[v] = nullptr;
    for (int v = 0; v < G.S; ++v) {
        if (!ptrs[v]) return fail(-1, "%s: NULL pointer for variable %d", what, v + 1);
        f.v[v] = ptrs[v];
    }
    return 0;
}

int require_ready() {
    if (!G.init) return fail(-4, "mfc_rhs_init has not been called");
    for (int d = 0; d < G.D; ++d)
        if (!G.dir[d].ready) return fail(-4, "mfc_rhs_set_grid has not been called for direction %d", d);
    return 0;
}

template <typename F>
int dispatch_nf_d(F &&f) {
    const int nf = G.prm.num_fluids, D = G.D;
#define MFC_CASE(NF, DD) \
    if (nf == NF && D == DD) return f(std::integral_constant<int, NF>{}, std::integral_constant<int, DD>{});
    MFC_CASE(1, 1) MFC_CASE(1, 2) MFC_CASE(1, 3)
    MFC_CASE(2, 1) MFC_CASE(2, 2) MFC_CASE(2, 3)
    MFC_CASE(3, 1) MFC_CASE(3, 2) MFC_CASE(3, 3)
    MFC_CASE(4, 1) MFC_CASE(4, 2) MFC_CASE(4, 3)
    MFC_CASE(5, 1) MFC_CASE(5, 2) MFC_CASE(5, 3)
    MFC_CASE(6, 1) MFC_CASE(6, 2) MFC_CASE(6, 3)
    MFC_CASE(7, 1) MFC_CASE(7, 2) MFC_CASE(7, 3)
    MFC_CASE(8, 1) MFC_CASE(8, 2) MFC_CASE(8, 3)
    MFC_CASE(9, 1) MFC_CASE(9, 2) MFC_CASE(9, 3)
    MFC_CASE(10, 1) MFC_CASE(10, 2) MFC_CASE(10, 3)
#undef MFC_CASE
    return fail(-1, "no kernels for num_fluids=%d, num_dims=%d", nf, D);
}

// prim: also the ghost cells' primitive values.
int bc_fill(const Fields &q, const Fields *prim = nullptr) {
    const Box x = box();
    const long n0 = (long)(2 * x.b) * (x.n + 1 + 2 * x.bj) * (x.p + 1 + 2 * x.bk);
    const long n1 = (long)(x.m + 1) * (2 * x.bj) * (x.p + 1 + 2 * x.bk);
    const long n2 = (long)(x.m + 1) * (x.n + 1) * (2 * x.bk);
    const long nmax = std::max(n0, std::max(n1, n2));
    const dim3 grid((unsigned)((nmax + 255) / 256), 1 + (G.D >= 2) + (G.D >= 3)), block(256);
    TimedScope ts(kKBcFill);
    const BcCodes bc{G.prm.bc_x_beg, G.prm.bc_x_end, G.prm.bc_y_beg, G.prm.bc_y_end, G.prm.bc_z_beg, G.prm.bc_z_end};
    if (prim)
        return dispatch_nf_d([&](auto NF, auto D) -> int {
            hipLaunchKernelGGL((k_bc_prim<decltype(NF)::value, decltype(D)::value>), grid, block, 0, G.stream, q, *prim,
                               eos(), x, bc, (unsigned)n0, (unsigned)n1, (unsigned)n2);
            HIPCHK(hipGetLastError());
            return 0;
        });
    hipLaunchKernelGGL(k_bc_fill, grid, block, 0, G.stream, q, G.S, G.prm.num_fluids, x, bc, (unsigned)n0, (unsigned)n1,
                       (unsigned)n2);
    HIPCHK(hipGetLastError());
    return 0;
}

int cons_to_prim_launch(const Fields &qc, const Fields &qp) {
    const Eos e = eos();
    TimedScope ts(kKConsToPrim);
    return dispatch_nf_d([&](auto NF, auto D) -> int {
        hipLaunchKernelGGL((k_cons_to_prim<decltype(NF)::value, decltype(D)::value>),
                           dim3((unsigned)((G.ng + 255) / 256)), dim3(256), 0, G.stream, qc, qp, e, G.ng);
        HIPCHK(hipGetLastError());
        return 0;
    });
}

// The coefficients (a CoefKind) that a kernel of directions d and e has.
int coef_kind(int d, int e) {
    return G.dir[d].canon && G.dir[e].canon ? kCanonCoef : G.dir[d].uniform && G.dir[e].uniform ? kEqualCoef : kCellCoef;
}

SweepArgs sweep_args(int d) {
    SweepArgs a;
    memset(&a, 0, sizeof a);
    a.coef = G.dir[d].coef;
    a.inv_ds = G.dir[d].inv_ds;
    a.eos = eos();
    a.eps = G.prm.weno_eps;
    a.nxg = G.nxg;
    a.nyg = G.nyg;
    a.ncell = G.dir[d].s + 2 * G.b + 1;
    a.m = G.prm.m;
    a.n = G.prm.n;
    a.p = G.prm.p;
    a.b = G.b;
    a.bj = G.prm.n > 0 ? G.b : 0;
    a.bk = G.prm.p > 0 ? G.b : 0;
    const int bcs[3][2] = {{G.prm.bc_x_beg, G.prm.bc_x_end}, {G.prm.bc_y_beg, G.prm.bc_y_end},
                           {G.prm.bc_z_beg, G.prm.bc_z_end}};
    a.bc_beg = bcs[d][0];
    a.bc_end = bcs[d][1];
    memcpy(a.bcs, bcs, sizeof bcs);
    a.uniform = coef_kind(d, d);
    for (int q = 0; q < kNCoef; ++q) {
        a.ucf[q] = G.dir[d].ucf[q];
        a.ucf32[q] = (float)G.dir[d].ucf[q];
    }
    if (d == 0) {
        // the launcher picks the uniform-coefficient kernels for WENO5 on uniform grids
        const bool uni = G.prm.weno_order == 5 && G.dir[0].uniform;
        const int tw = G.prm.precision == MFC_PREC_FP32_LEARNED ? x_tile_cells<true, float, true>()
                       : G.prm.precision == MFC_PREC_FP32_BULK
                           ? (uni ? x_tile_cells<false, float, true>() : x_tile_cells<false, float, false>())
                           : (uni ? x_tile_cells<false, double, true>() : x_tile_cells<false, double, false>());
        a.ntile = (G.prm.m + 1 + tw - 1) / tw;
        a.nblocks = (long)a.ntile * (G.prm.n + 1) * (G.prm.p + 1);
    } else {
        const int s = G.dir[d].s;
        const bool uni = G.prm.weno_order == 5 && G.dir[d].uniform;
        const bool cp = G.prm.precision == MFC_PREC_FP32_LEARNED ? t_cell_parallel<true, float, true>()
                        : G.prm.precision == MFC_PREC_FP32_BULK
                            ? (uni ? t_cell_parallel<false, float, true>() : t_cell_parallel<false, float, false>())
                            : (uni ? t_cell_parallel<false, double, true>() : t_cell_parallel<false, double, false>());
        const bool f64 = G.prm.precision == MFC_PREC_FP64 || G.prm.precision == MFC_PREC_FP64_FAST;
        const int xc = !cp ? kTX : tc_cols_of(G.prm.precision == MFC_PREC_FP32_LEARNED, d);
        a.ntile = (G.prm.m + 1 + xc - 1) / xc;
        a.chunk = G.prm.precision == MFC_PREC_FP32_LEARNED ? t_tile_cells<true, float, true>(d)
                  : G.prm.precision == MFC_PREC_FP32_BULK
                      ? (uni ? t_tile_cells<false, float, true>(d) : t_tile_cells<false, float, false>(d))
                  : !uni ? t_tile_cells<false, double, false>(d)
                         : tc_rows_of(true, G.prm.precision == MFC_PREC_FP64_FAST, d) - 2;
        a.nchunk = (s + 1 + a.chunk - 1) / a.chunk;
        const int other = d == 1 ? G.prm.p + 1 : G.prm.n + 1;
        a.nblocks = (long)a.ntile * a.nchunk * other;
    }
    return a;
}

// Arguments of the fused x and y sweep: the x direction's, the y
// direction's cell widths, boundary codes and coefficients, and its tiles.
SweepArgs xy_args() {
    SweepArgs a = sweep_args(0);
    a.uniform = coef_kind(0, 1);
    a.inv_ds2 = G.dir[1].inv_ds;
    a.bc2_beg = G.prm.bc_y_beg;
    a.bc2_end = G.prm.bc_y_end;
    for (int q = 0; q < kNCoef; ++q) {
        a.ucf2[q] = G.dir[1].ucf[q];
        a.ucf2_32[q] = (float)G.dir[1].ucf[q];
    }
    a.ntile = (G.prm.m + 1 + kXyCellsX - 1) / kXyCellsX;
    a.nchunk = (G.prm.n + 1 + kXyCellsY - 1) / kXyCellsY;
    a.nblocks = (long)a.ntile * a.nchunk * (G.prm.p + 1);
    return a;
}

// Arguments of a march (k_march): d = 4 the y march with the x faces, d = 5
// the z march, d = 7 the y march alone.
SweepArgs march_args(int d) {
    SweepArgs a = d == 4 ? xy_args() : sweep_args(d == 5 ? 2 : 1);
    const int cells = d == 4 ? kMarchCellsXY : kMarchCellsZ, rows = d == 5 ? G.prm.p + 1 : G.prm.n + 1;
    const int other = d == 5 ? G.prm.n + 1 : G.prm.p + 1;
    if (d == 4) {
        a.coef2 = G.dir[1].coef;
        a.ncell2 = G.dir[1].s + 2 * G.b + 1;
    }
    a.rl = d == 4 ? G.prm.m + 1 + 2 * kMarchHaloXY : G.prm.m + 1;
    a.ntile = (int)(((long)a.rl * other + cells - 1) / cells);
    // Chunks of rows: a chunk costs three rows more than it finishes (the
    // staged rows and the reconstructions before its first face).
    const int slots = G.prm.precision == MFC_PREC_FP32_BULK ? kMarchSlots32 : kMarchSlots;
    double best = 0.0;
    for (int nc = 1; nc <= rows; ++nc) {
        const int L = (rows + nc - 1) / nc;
        if (L < kMarchChunkMin && nc > 1) break;
        if ((rows + L - 1) / L != nc) continue;
        const double cost = chunk_rounds((double)a.ntile * nc, slots) * (L + 3);
        if (best == 0.0 || cost < best) best = cost, a.chunk = L, a.nchunk = nc;
    }
    a.nblocks = (long)a.ntile * a.nchunk;
    return a;
}

// Whether the x and y directions (d = 4), the z direction (d = 5) or with
// three fluids the y direction (d = 7) of a WENO5 case of the plain,
// contracted or FP32-bulk form run as a march.
bool marches(int d) {
    if (G.visc || G.prm.precision == MFC_PREC_FP32_LEARNED || G.prm.weno_order != 5 ||
        G.prm.num_fluids > (d == 4 ? kMarchMaxFluidsXY : kMarchMaxFluidsZ) ||
        (d == 7 && G.prm.num_fluids <= kMarchMaxFluidsXY) || G.D < (d == 4 ? 2 : 3))
        return false;
    if (G.ng * (long)sizeof(double) >= (1L << 32)) return false; // 32-bit byte offsets within a variable
    const bool uni = d == 4 ? G.dir[0].uniform && G.dir[1].uniform : G.dir[d == 5 ? 2 : 1].uniform;
    if (uni && (d == 7 || G.prm.precision == MFC_PREC_FP32_BULK)) return false;
    if (d == 7 && G.prm.precision == MFC_PREC_FP32_BULK) return false;
    if ((double)G.nint < (!uni ? kMarchPerCell : G.D == 2 ? kMarchUniform2D : kMarchUniform3D)) return false;
    // short rows or few of them: the lanes and rows a march adds at the ends
    // would outweigh what it saves
    const SweepArgs a = march_args(d);
    const int rows = d == 5 ? G.prm.p + 1 : G.prm.n + 1;
    return rows >= kMarchRowsMin &&
           (double)G.nint / rows >= 0.85 * a.ntile * (d == 4 ? kMarchCellsXY : kMarchCellsZ);
}

// Arguments of k_rows_x.
SweepArgs rows_args() {
    SweepArgs a = sweep_args(0);
    a.rl = G.prm.m + 7;
    a.ntile = (int)(((long)a.rl * (G.prm.p + 1) + kRowsCells - 4) / kRowsCells);
    // Chunks as in march_args; a chunk costs about half a row more than it
    // finishes (the coefficients' loads).  Past one round the launch's time
    // grows in half rounds, one wave more per SIMD each (16 grids with 1 to 13
    // rows a chunk: 1.41 rounds' time for 1.06 rounds of waves, 1.47 for 1.49,
    // 1.85 for 1.59, 2.32 for 2.22).
    const int rows = G.prm.n + 1;
    double best = 0.0;
    for (int L = 1; L <= std::min(rows, 32); ++L) {
        const int nc = (rows + L - 1) / L;
        const double r = (double)a.ntile * nc / kMarchSlots;
        const double cost = (r <= 1.0 ? 1.0 : 0.1 + 0.45 * std::ceil(2.0 * r)) * (L + 0.5);
        if (best == 0.0 || cost < best) best = cost, a.chunk = L, a.nchunk = nc;
    }
    a.nblocks = (long)a.ntile * a.nchunk;
    return a;
}

// Whether the x direction of a case on unequal widths runs along rows
// (k_rows_x): from two rounds of waves with a row each, and where the x sweep's
// waves (63 cells each, four per SIMD) do not all have a place at once.  RK3
// step, plain or contracted (c), x sweep -> rows: 600 x 500 cells (5500 sets of
// columns and rows) 188 -> 179 us, 700 x 700 269 -> 245, 1000 x 900 411 -> 388, c
// 800 x 800 214 -> 205; 96^3 750 -> 696; three fluids c 180 x 130 x 90 1806 ->
// 1221, plain 2349 -> 1841.  Just above the line 64 x 69 x 51 (4278 sets, 7038
// waves of the x sweep; RK2) 210 -> 178; where the x sweep has fewer than 4096
// waves rows took 0.97 to 1.06 of its time (57 x 82 x 48 185 -> 191).
constexpr long kRowsMin = 2 * kMarchSlots, kSweepXSlots = 16 * 256;
bool rows_x() {
    if (G.D < 2 || G.visc || G.prm.weno_order != 5 || G.prm.num_fluids > kRowsMaxFluids || G.dir[0].uniform ||
        (G.prm.precision != MFC_PREC_FP64 && G.prm.precision != MFC_PREC_FP64_FAST))
        return false;
    if (G.ng * (long)sizeof(double) >= (1L << 32)) return false; // 32-bit byte offsets within a variable
    return sweep_args(0).nblocks > kSweepXSlots && (long)rows_args().ntile * (G.prm.n + 1) >= kRowsMin;
}

// Arguments of k_stage.
SweepArgs stage_args() {
    SweepArgs a = G.D == 2 ? xy_args() : sweep_args(0);
    if (G.D == 2) {
        a.coef2 = G.dir[1].coef;
        a.ncell2 = G.dir[1].s + 2 * G.b + 1;
    }
    a.ntile = (G.prm.m + stage_cells_x(G.D)) / stage_cells_x(G.D);
    a.nblocks = (long)a.ntile * ((G.prm.n + stage_cells_y(G.D)) / stage_cells_y(G.D));
    return a;
}

// Whether an RK stage runs as one kernel (k_stage).  In 2D as long as every
// block has a compute unit of its own: RK3 step on 256 x 160 cells (256
// blocks) 66.5 -> 48.1 us, contracted 45.5 -> 38.5 us, but on 256 x 170 cells
// 66.2 -> 74.3 us.  In 1D blocks share compute units: 1000 cells 29.1 -> 24.3
// us, 100000 cells 34.9 -> 32.5 us and contracted level, 28.3 and 28.0 us.
constexpr long kStageBlocks2D = 256, kStageBlocks1D = 1600;
bool stage_in_one() {
    return G.D <= 2 && !G.visc && G.prm.weno_order == 5 && G.prm.num_fluids <= kXyMaxFluids &&
           (G.prm.precision == MFC_PREC_FP64 || G.prm.precision == MFC_PREC_FP64_FAST) &&
           stage_args().nblocks <= (G.D == 2 ? kStageBlocks2D : kStageBlocks1D);
}

// d = 0, 1, 2: one direction; d = 3: the fused x and y sweep; d = 4, 5: the
// marches; d = 6: an RK stage in one kernel; d = 7: the y march.
int sweep(int d, SweepArgs &a) {
    SweepLaunch L{d, G.D, G.prm.weno_order, G.prm.precision};
    if (G.prm.precision == MFC_PREC_FP32_LEARNED) {
        a.mlp = mlp_frags();
        if (!a.mlp) return fail(-4, "learned weights requested but mfc_mlp_init has not been called");
    }
    static constexpr int kinds[] = {kKSweepX, kKSweepX + 1, kKSweepX + 2, kKSweepXY, kKSweepXY, kKSweepZ, kKSweepXY,
                                    kKSweepX + 1, kKSweepX};
    static constexpr int subs[] = {-1, -1, -1, kKTileXY, kKMarchXY, kKMarchZ, kKStage, kKMarchY, kKRowsX};
    TimedScope ts(d == 6 && G.D == 1 ? kKSweepX : kinds[d], subs[d]);
    int rc;
    const int form = G.prm.precision == MFC_PREC_FP64        ? kFormF64
                     : G.prm.precision == MFC_PREC_FP64_FAST ? kFormF64Fast
                                                             : kFormF32;
    auto go = [&](auto nf) -> int {
        constexpr int NF = decltype(nf)::value;
        if (form == kFormF64) return launch_sweep<NF, kFormF64>(L, a, G.stream);
        if (form == kFormF64Fast) return launch_sweep<NF, kFormF64Fast>(L, a, G.stream);
        if constexpr (NF <= kNumFluidsBuiltF32) return launch_sweep<NF, kFormF32>(L, a, G.stream);
        return -1;
    };
    switch (G.prm.num_fluids) {
    case 1: rc = go(std::integral_constant<int, 1>{}); break;
    case 2: rc = go(std::integral_constant<int, 2>{}); break;
    case 3: rc = go(std::integral_constant<int, 3>{}); break;
    case 4: rc = go(std::integral_constant<int, 4>{}); break;
    case 5: rc = go(std::integral_constant<int, 5>{}); break;
    case 6: rc = go(std::integral_constant<int, 6>{}); break;
    case 7: rc = go(std::integral_constant<int, 7>{}); break;
    case 8: rc = go(std::integral_constant<int, 8>{}); break;
    case 9: rc = go(std::integral_constant<int, 9>{}); break;
    case 10: rc = go(std::integral_constant<int, 10>{}); break;
    default: rc = -1;
    }
    if (rc != 0) return fail(-3, "sweep launch failed (dir %d): %s", d, hipGetErrorString(hipGetLastError()));
    return 0;
}

// Direction d of a viscous RHS evaluation (inviscid and viscous fluxes of
// every face, then the finish: m_rhs.fpp:565-652), with sa the direction's
// finish arguments (rhs assignment or accumulation, or the RK stage).
int viscous(int d, const Fields &qin, const SweepArgs &sa) {
    ViscArgs v;
    memset(&v, 0, sizeof v);
    v.q = qin;
    v.coef = G.dir[d].coef;
    v.ncell = G.dir[d].s + 2 * G.b + 1;
    v.uniform = G.dir[d].uniform ? 1 : 0;
    for (int q = 0; q < kNCoef; ++q) v.ucf[q] = G.dir[d].ucf[q];
    v.ccx = G.dir[0].cc_dev;
    v.ccy = G.D > 1 ? G.dir[1].cc_dev : nullptr;
    v.inv_ds = G.dir[d].inv_ds;
    v.eos = eos();
    v.eps = G.prm.weno_eps;
    v.nxg = G.nxg;
    v.m = G.prm.m;
    v.n = G.prm.n;
    v.b = G.b;
    v.bj = G.prm.n > 0 ? G.b : 0;
    const int bcs[2][2] = {{G.prm.bc_x_beg, G.prm.bc_x_end}, {G.prm.bc_y_beg, G.prm.bc_y_end}};
    v.bc_beg = bcs[d][0];
    v.bc_end = bcs[d][1];
    v.vp = G.vp;
    v.grad = G.visc_grad;
    v.ng = G.ng;
    v.wrf = G.wrf ? 1 : 0;
    TimedScope ts(kKViscous);
    if (launch_viscous(G.prm.num_fluids, G.D, d, G.prm.weno_order, v, sa, G.stream))
        return fail(-3, "viscous launch failed (dir %d): %s", d, hipGetErrorString(hipGetLastError()));
    return 0;
}

// Whether the sweep that writes an RK stage fills the stage's ghost cells.
bool sweeps_fill_ghosts() {
    if (G.visc || G.D > 2) return false;
    if (G.D == 1 || G.prm.precision == MFC_PREC_FP32_LEARNED) return true;
    return G.prm.precision != MFC_PREC_FP32_BULK && kFuseXY && G.prm.weno_order == 5 &&
           G.prm.num_fluids <= kXyMaxFluids && G.dir[0].uniform && G.dir[1].uniform && !marches(4);
}

// Whether the x and y march can store the primitive field of its input.
bool march_stores_prim() { return G.prm.precision == MFC_PREC_FP64 && kFuseXY && marches(4); }

// All directional sweeps of one RHS evaluation on the ghost-filled field qin.
// The last sweep either writes rhs (rk = kRkNone) or applies the RK stage.
// Viscous runs use the viscous kernels for each direction instead, with the
// same finish semantics.
// ghosts: the last sweep also fills the ghost cells of *qout (the caller's
// next stage input; sweeps_fill_ghosts).
// prim: the x and y march also stores the interior's primitive values
// (march_stores_prim).
int sweeps(const Fields &qin, const Fields &rhs, int rk, const Fields *qbase, const Fields *qout, double dt,
           bool ghosts = false, const Fields *prim = nullptr) {
    // The plain form adds the directions in the reference's order x, y, z
    // (m_rhs.fpp:469-656; it fixes the rounding).  The contracted FP64,
    // FP32-bulk and learned forms run them in the reverse order: the sum is
    // the same up to rounding, and the RK stage's output is then written by
    // the x sweep (or the fused x and y sweep), whose loads are contiguous
    // rows (learned form, 512^3: 68.2 -> 64.5 ms per step, 2048^2 1.47 ->
    // 1.35 ms).
    const bool reverse = (G.prm.precision == MFC_PREC_FP64_FAST || G.prm.precision == MFC_PREC_FP32_BULK ||
                          G.prm.precision == MFC_PREC_FP32_LEARNED) &&
                         !G.visc;
    if (G.wrf) {
        // cell-centred velocity gradients of the stage input (s_get_viscous,
        // m_rhs.fpp:456-464), before the directions
        ViscGradArgs g;
        memset(&g, 0, sizeof g);
        g.q = qin;
        g.grad = G.visc_grad;
        g.eps = G.prm.weno_eps;
        g.nxg = G.nxg;
        g.ng = G.ng;
        g.b = G.b;
        g.uniform = 1;
        for (int e = 0; e < G.D; ++e) {
            g.coef[e] = G.dir[e].coef;
            g.ncell[e] = G.dir[e].s + 2 * G.b + 1;
            g.inv_dsg[e] = G.dir[e].inv_dsg;
            g.s[e] = G.dir[e].s;
            g.uniform &= G.dir[e].uniform_wide ? 1 : 0;
            for (int q = 0; q < kNCoef; ++q) g.ucf[e][q] = G.dir[e].ucf[q];
        }
        TimedScope ts(kKViscous);
        if (launch_visc_grad(G.prm.num_fluids, G.D, G.prm.weno_order, g, G.stream))
            return fail(-3, "viscous gradient launch failed: %s", hipGetErrorString(hipGetLastError()));
    }
    // The contracted form spreads an RK stage over its sweeps (out = cb*base
    // + ci*in + cdt*L; the sweeps before the last read the base, the last
    // the stage input's own cells, which it stages anyway), so the x sweep
    // does not carry a fourth array.
    const bool fold = reverse && rk != kRkNone && G.D > 1;
    double cb = 1.0, ci = 0.0, cdt = dt;
    if (rk == kRk2Final) {
        cb = 0.5, ci = 0.5, cdt = 0.5 * dt;
    } else if (rk == kRk3Stage2) {
        cb = 0.75, ci = 0.25, cdt = 0.25 * dt;
    } else if (rk == kRk3Stage3) {
        cb = 1.0 / 3.0, ci = 2.0 / 3.0, cdt = 2.0 * dt / 3.0;
    }
    if (fold && qbase->v[0] == qin.v[0]) {
        // base = in (first stages): (cb + ci)*in, added by the last sweep
        // from its staged cells, and no sweep reads the base
        ci += cb;
        cb = 0.0;
    }
    // The contracted and FP32-bulk forms, WENO5, one or two fluids, fuse the y
    // and x sweeps on grids uniform in x and y (k_sweep_xy) or large enough for
    // a march (k_march): in 3D after the z sweep, in 2D alone.
    const bool march = marches(4), marchz = marches(5), marchy = marches(7);
    const bool fuse = reverse && kFuseXY && G.D >= 2 &&
                      (G.prm.precision == MFC_PREC_FP64_FAST || G.prm.precision == MFC_PREC_FP32_BULK) &&
                      G.prm.weno_order == 5 && G.prm.num_fluids <= kXyMaxFluids &&
                      (march || (G.dir[0].uniform && G.dir[1].uniform));
    if (fuse) {
        const int split = G.D == 3 ? std::min(kBaseOnZFused, G.S) : 0;
        auto stage = [&](SweepArgs &a, int fold_kind, int lo, int hi) {
            a.qin = qin;
            a.rhs = rhs;
            a.dt = dt;
            a.rk = kRkNone;
            a.ghosts = ghosts && fold_kind == 3;
            if (fold) {
                a.qbase = *qbase;
                a.qout = *qout;
                a.base_is_in = qbase->v[0] == qin.v[0];
                a.fold = fold_kind;
                if (cb != 0.0) a.base_lo = lo, a.base_hi = hi;
                a.cb = cb;
                a.ci = ci;
                a.cdt = cdt;
            }
        };
        if (G.D == 3) {
            SweepArgs a = marchz ? march_args(5) : sweep_args(2);
            stage(a, 1, 0, split);
            a.accumulate = 0;
            if (int rc = sweep(marchz ? 5 : 2, a)) return rc;
        }
        SweepArgs a = march ? march_args(4) : xy_args();
        stage(a, 3, split, G.S);
        a.accumulate = G.D == 3;
        return sweep(march ? 4 : 3, a);
    }
    // The plain form fuses its first two directions the same way (bitwise
    // the separate x and y sweeps): in 3D the z sweep then adds its part and
    // applies the RK stage, in 2D the fused sweep applies it.
    const bool fuse_plain = kFuseXY && !G.visc && G.D >= 2 && G.prm.precision == MFC_PREC_FP64 &&
                            G.prm.weno_order == 5 && G.prm.num_fluids <= kXyMaxFluids &&
                            (march || (G.dir[0].uniform && G.dir[1].uniform));
    if (fuse_plain) {
        auto finish = [&](SweepArgs &a, bool last) {
            a.qin = qin;
            a.rhs = rhs;
            a.dt = dt;
            a.rk = last ? rk : kRkNone;
            a.ghosts = ghosts && last;
            if (a.rk != kRkNone) {
                a.qbase = *qbase;
                a.qout = *qout;
                a.base_is_in = qbase->v[0] == qin.v[0];
            }
        };
        SweepArgs a = march ? march_args(4) : xy_args();
        finish(a, G.D == 2);
        a.accumulate = 0;
        if (prim) a.prim = *prim;
        if (int rc = sweep(march ? 4 : 3, a)) return rc;
        if (G.D == 3) {
            SweepArgs z = marchz ? march_args(5) : sweep_args(2);
            finish(z, true);
            z.accumulate = 1;
            return sweep(marchz ? 5 : 2, z);
        }
        return 0;
    }
    for (int k = 0; k < G.D; ++k) {
        const int d = reverse ? G.D - 1 - k : k;
        const int ld = d == 2 && marchz ? 5 : d == 1 && marchy ? 7 : d == 0 && rows_x() ? 8 : d;
        SweepArgs a = ld == d ? sweep_args(d) : ld == 8 ? rows_args() : march_args(ld);
        a.qin = qin;
        a.rhs = rhs;
        a.accumulate = k > 0;
        a.dt = dt;
        const bool last = k == G.D - 1;
        a.rk = last && !fold ? rk : kRkNone;
        a.ghosts = ghosts && last;
        if (a.rk != kRkNone || fold) {
            a.qbase = *qbase;
            a.qout = *qout;
            a.base_is_in = qbase->v[0] == qin.v[0];
        }
        if (fold) {
            a.fold = k == 0 ? 1 : last ? 3 : 2;
            // cb*base: in 3D variables [0, kBaseOnZ) on the z sweep, the rest
            // on y; in 2D all on y (the first sweep)
            const int split = G.D == 3 ? marchz || marchy ? kBaseOnZFused : kBaseOnZ : 0;
            if (cb != 0.0 && k == 0 && G.D == 3) a.base_lo = 0, a.base_hi = split;
            if (cb != 0.0 && k == G.D - 2) a.base_lo = split, a.base_hi = G.S;
            a.cb = cb;
            a.ci = ci;
            a.cdt = cdt;
        }
        if (int rc = G.visc ? viscous(d, qin, a) : sweep(ld, a)) return rc;
    }
    return 0;
}

} // namespace

// ===========================================================================
// C ABI

extern "C" {

const char *mfc_last_error(void) { return g_err.c_str(); }

int mfc_rhs_init(const mfc_params *prm) {
    if (!prm) return fail(-1, "NULL params");
    if (int rc = check_params(*prm)) return rc;
    if (G.init) mfc_rhs_finalize();
    G.prm = *prm;
    G.D = 1 + (prm->n > 0) + (prm->p > 0);
    G.S = 2 * prm->num_fluids + G.D + 1;
    G.polyn = (prm->weno_order - 1) / 2;
    // buff_size (m_global_parameters.fpp:355-359): viscous cases keep
    // 2*polyn + 2 ghost layers, inviscid ones polyn + 2
    bool visc = false;
    for (int i = 0; i < prm->num_fluids; ++i)
        for (int r = 0; r < 2; ++r) visc = visc || prm->Re[i][r] > 0.0;
    G.b = visc ? 2 * G.polyn + 2 : G.polyn + 2;
    G.nxg = prm->m + 2 * G.b + 1;
    G.nyg = prm->n > 0 ? prm->n + 2 * G.b + 1 : 1;
    G.nzg = prm->p > 0 ? prm->p + 2 * G.b + 1 : 1;
    G.ng = G.nxg * G.nyg * G.nzg;
    // The sweeps address a block's cells as a uniform base plus a 32-bit
    // byte offset per lane (Off in mfc_sweep.hpp); a z-sweep block spans at
    // most 40 ghosted planes
    if (G.nzg > 1 && 40L * G.nxg * G.nyg * (long)sizeof(double) >= (1L << 32))
        return fail(-1, "a z plane of %ld x %ld ghosted cells exceeds the sweeps' 32-bit block offsets", (long)G.nxg,
                    (long)G.nyg);
    G.nint = (long)(prm->m + 1) * (prm->n + 1) * (prm->p + 1);
    G.dir[0].s = prm->m;
    G.dir[1].s = prm->n;
    G.dir[2].s = prm->p;
    HIPCHK(hipStreamCreateWithFlags(&G.own, hipStreamNonBlocking));
    G.stream = G.own;
    HIPCHK(hipMalloc(&G.partials, sizeof(double) * 2 * kReduceBlocks));
    if (!g_result) HIPCHK(hipHostMalloc(&g_result, sizeof(double), hipHostMallocPortable));
    {
        int dev = 0;
        HIPCHK(hipGetDevice(&dev));
        if (dev < 0 || dev >= kMaxDevices) return fail(-3, "device ordinal %d outside 0..%d", dev, kMaxDevices - 1);
        if (!g_scratch_dev[dev]) {
            void *ptr = nullptr;
            HIPCHK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
            g_scratch_dev[dev] = static_cast<double *>(ptr);
            HIPCHK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(icfl_done)));
            g_done_dev[dev] = static_cast<unsigned *>(ptr);
        }
        G.scratch = g_scratch_dev[dev];
        G.count = g_done_dev[dev];
    }
    // Re_size, Re_idx, Res (m_global_parameters.fpp:314-338, m_viscous.fpp:36-42)
    for (int r = 0; r < 2; ++r)
        for (int i = 0; i < prm->num_fluids; ++i)
            if (prm->Re[i][r] > 0.0) {
                G.vp.idx[r][G.vp.size[r]] = i;
                G.vp.res[r][G.vp.size[r]] = prm->Re[i][r];
                G.vp.size[r]++;
            }
    G.visc = G.vp.size[0] > 0 || G.vp.size[1] > 0;
    if (G.visc) {
        G.wrf = prm->weno_Re_flux != 0;
        if (G.wrf) HIPCHK(hipMalloc(&G.visc_grad, sizeof(double) * G.D * G.D * G.ng));
    }
    G.init = true;
    return 0;
}

int mfc_rhs_set_grid(int dir, const double *s_cb, const double *ds) {
    if (!G.init) return fail(-4, "mfc_rhs_init has not been called");
    if (dir < 0 || dir >= G.D) return fail(-1, "direction %d outside 0..%d", dir, G.D - 1);
    if (!s_cb || !ds) return fail(-1, "NULL grid array");
    Dir &D = G.dir[dir];
    const int s = D.s, b = G.b;
    for (int i = 0; i <= s; ++i)
        if (!(ds[i + b] > 0.0)) return fail(-1, "non-positive cell width at index %d of direction %d", i, dir);
    weno_tables(s, b, G.prm.weno_order, s_cb, D.coef_h);
    // Uniform coefficients over the cells the sweeps reconstruct (-1..s+1)?
    // Bit for bit in the plain FP64 form; within kUniformRelTol of cell -1's
    // in the others, whose uniform-grid kernels then use cell -1's (but see
    // canon).
    {
        const long nc = s + 2 * b + 1;
        const double tol = G.prm.precision == MFC_PREC_FP64 ? 0.0 : kUniformRelTol;
        D.uniform = true;
        for (int q = 0; q < kNCoef && D.uniform; ++q) {
            const double v0 = D.coef_h[(long)q * nc + (-1 + b)];
            D.ucf[q] = v0;
            for (int j = 0; j <= s + 1 && D.uniform; ++j) {
                const double v = D.coef_h[(long)q * nc + (j + b)];
                D.uniform = std::memcmp(&v0, &v, sizeof(double)) == 0 || std::fabs(v - v0) <= tol * std::fabs(v0);
            }
        }
    }
    // The contracted form has WENO5 kernels with the constants of equal cell
    // widths built in (weno5_canon), for cells that all lie within the same
    // tolerance of those.  Equal coefficients of unequal widths (a geometric
    // grid) keep cell -1's: with each cell's own, 1024^2 cells took 311 instead
    // of 234 us per step, 64^3 204 instead of 170.
    D.canon = D.uniform && G.prm.precision == MFC_PREC_FP64_FAST && G.prm.weno_order == 5;
    for (int q = 0; q < kNCoef && D.canon; ++q) {
        const double *c = &D.coef_h[(long)q * (s + 2 * b + 1) + (b - 1)], at = kCanon[q];
        const double tol = kUniformRelTol * std::fabs(at);
        int far = 0;
        for (int j = 0; j < s + 3; ++j) far |= !(std::fabs(c[j] - at) <= tol);
        D.canon = !far;
    }
    // Uniform over every cell with coefficients (the weno_Re_flux gradient
    // pass reconstructs the ghost cells too)?
    {
        const long nc = s + 2 * b + 1;
        const int pn = (G.prm.weno_order - 1) / 2;
        D.uniform_wide = D.uniform;
        for (int q = 0; q < kNCoef && D.uniform_wide; ++q)
            for (int j = -b + pn; j <= s + b - pn && D.uniform_wide; ++j)
                D.uniform_wide = std::memcmp(&D.ucf[q], &D.coef_h[(long)q * nc + (j + b)], sizeof(double)) == 0;
    }
    std::vector<double> inv(s + 1), invg(s + 2 * b + 1);
    for (int i = 0; i <= s; ++i) inv[i] = 1.0 / ds[i + b];
    for (int i = -b; i <= s + b; ++i) invg[i + b] = 1.0 / ds[i + b]; // 1d0/dx(j), m_viscous.fpp:386-393
    // cell centres with ghosts (m_start_up.fpp:356-359, :551, :582)
    std::vector<double> cc(s + 2 * b + 1);
    for (int i = 0; i <= s; ++i) cc[i + b] = s_cb[i - 1 + 1 + b] + ds[i + b] / 2.0;
    for (int i = 1; i <= b; ++i) cc[-i + b] = cc[1 - i + b] - (ds[1 - i + b] + ds[-i + b]) / 2.0;
    for (int i = 1; i <= b; ++i) cc[s + i + b] = cc[s + (i - 1) + b] + (ds[s + (i - 1) + b] + ds[s + i + b]) / 2.0;
    D.ds_h.assign(ds, ds + s + 2 * b + 1);
    if (D.coef) HIPCHK(hipFree(D.coef));
    if (D.inv_ds) HIPCHK(hipFree(D.inv_ds));
    if (D.ds_dev) HIPCHK(hipFree(D.ds_dev));
    if (D.cc_dev) HIPCHK(hipFree(D.cc_dev));
    if (D.inv_dsg) HIPCHK(hipFree(D.inv_dsg));
    D.inv_dsg = nullptr;
    D.coef = nullptr;
    D.inv_ds = nullptr;
    D.ds_dev = nullptr;
    D.cc_dev = nullptr;
    HIPCHK(hipMalloc(&D.coef, sizeof(double) * D.coef_h.size()));
    HIPCHK(hipMalloc(&D.inv_ds, sizeof(double) * inv.size()));
    HIPCHK(hipMalloc(&D.ds_dev, sizeof(double) * (s + 1)));
    HIPCHK(hipMalloc(&D.cc_dev, sizeof(double) * cc.size()));
    HIPCHK(hipMemcpy(D.cc_dev, cc.data(), sizeof(double) * cc.size(), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(D.ds_dev, ds + b, sizeof(double) * (s + 1), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(D.coef, D.coef_h.data(), sizeof(double) * D.coef_h.size(), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(D.inv_ds, inv.data(), sizeof(double) * inv.size(), hipMemcpyHostToDevice));
    if (G.wrf) {
        HIPCHK(hipMalloc(&D.inv_dsg, sizeof(double) * invg.size()));
        HIPCHK(hipMemcpy(D.inv_dsg, invg.data(), sizeof(double) * invg.size(), hipMemcpyHostToDevice));
    }
    D.ready = true;
    return 0;
}

int mfc_compute_rhs(double *const *q_cons_vf, double *const *q_prim_vf, double *const *rhs_vf, int t_step) {
    if (int rc = require_ready()) return rc;
    Fields qc, qp, rhs;
    if (int rc = fields(q_cons_vf, qc, "q_cons_vf")) return rc;
    // the primitive field from the march that converts the cells anyway
    const bool fused = q_prim_vf && t_step != G.prm.t_step_stop && march_stores_prim();
    if (!fused)
        if (int rc = bc_fill(qc)) return rc;
    if (t_step == G.prm.t_step_stop) return 1;
    if (int rc = fields(rhs_vf, rhs, "rhs_vf")) return rc;
    if (q_prim_vf) {
        if (int rc = fields(q_prim_vf, qp, "q_prim_vf")) return rc;
        if (int rc = fused ? bc_fill(qc, &qp) : cons_to_prim_launch(qc, qp)) return rc;
    }
    if (fused) return sweeps(qc, rhs, kRkNone, nullptr, nullptr, 0.0, false, &qp);
    return sweeps(qc, rhs, kRkNone, nullptr, nullptr, 0.0);
}

int mfc_tvd_rk_step(int t_step, double dt, double *const *q_cons_ts1, double *const *q_cons_ts2,
                    double *const *q_prim_vf, double *const *rhs_vf) {
    if (int rc = require_ready()) return rc;
    Fields q1, q2, qp, rhs;
    if (int rc = fields(q_cons_ts1, q1, "q_cons_ts(1)")) return rc;
    if (int rc = fields(rhs_vf, rhs, "rhs_vf")) return rc;
    if (G.prm.time_stepper > 1)
        if (int rc = fields(q_cons_ts2, q2, "q_cons_ts(2)")) return rc;
    // each stage in one kernel, which reads its input's ghost cells through the
    // boundary codes; it fills them only in the caller's arrays
    const bool one = G.prm.time_stepper > 1 && stage_in_one();
    if (!one || q_prim_vf || t_step == G.prm.t_step_stop)
        if (int rc = bc_fill(q1)) return rc;
    if (t_step == G.prm.t_step_stop) return 1;
    if (q_prim_vf) {
        if (int rc = fields(q_prim_vf, qp, "q_prim_vf")) return rc;
        if (int rc = cons_to_prim_launch(q1, qp)) return rc;
    }
    if (G.prm.time_stepper == 1) {
        if (int rc = sweeps(q1, rhs, kRkNone, nullptr, nullptr, dt)) return rc;
        const Box x = box();
        TimedScope ts(kKRk1);
        hipLaunchKernelGGL(k_rk1_update, dim3((unsigned)((G.nint + 255) / 256)), dim3(256), 0, G.stream, q1, rhs,
                           G.S, x, dt, G.nint);
        HIPCHK(hipGetLastError());
        return 0;
    }
    // a stage whose output is the next stage's input, with its ghost cells
    const bool filled = sweeps_fill_ghosts();
    auto stage = [&](const Fields &in, int rk, const Fields &out) -> int {
        if (one) {
            SweepArgs a = stage_args();
            a.qin = in;
            a.qbase = q1;
            a.qout = out;
            a.dt = dt;
            a.rk = rk;
            a.ghosts = in.v[0] != G.scratch_state;
            return sweep(6, a);
        }
        const bool next = out.v[0] != q1.v[0]; // another stage follows
        if (int rc = sweeps(in, rhs, rk, &q1, &out, dt, filled && next)) return rc;
        return filled || !next ? 0 : bc_fill(out);
    };
    if (G.prm.time_stepper == 2) {
        if (int rc = stage(q1, kRkEuler, q2)) return rc;
        return stage(q2, kRk2Final, q1);
    }
    if (!G.scratch_state) HIPCHK(hipMalloc(&G.scratch_state, sizeof(double) * G.S * G.ng));
    Fields q3;
    for (int v = 0; v < kMaxSys; ++v) q3.v[v] = v < G.S ? G.scratch_state + (long)v * G.ng : nullptr;
    // stage 1: q3 = q1 + dt*L(q1); stage 2: q2 = (3 q1 + q3 + dt*L(q3))/4;
    // stage 3: q1 = (q1 + 2 q2 + 2 dt*L(q2))/3.  Each stage reads its input's
    // stencil and writes a different array, or only its own cell of q1.
    if (int rc = stage(q1, kRkEuler, q3)) return rc;
    if (int rc = stage(q3, kRk3Stage2, q2)) return rc;
    return stage(q2, kRk3Stage3, q1);
}

int mfc_cons_to_prim(double *const *q_cons_vf, double *const *q_prim_vf) {
    if (!G.init) return fail(-4, "mfc_rhs_init has not been called");
    Fields qc, qp;
    if (int rc = fields(q_cons_vf, qc, "q_cons_vf")) return rc;
    if (int rc = fields(q_prim_vf, qp, "q_prim_vf")) return rc;
    return cons_to_prim_launch(qc, qp);
}

// The ICFL max-reduction into `partials` (capacity doubles), a grid-stride
// pass of at most kCflBlocks blocks, so every grid size fits.  `timed`
// records HIP events around the pass (event creation may allocate, so the
// allocation-free entry point passes false).  The caller holds g_reduce.
static int icfl_reduce(double *const *q, bool from_cons, double dt, double *out, double *partials, int capacity,
                       bool timed) {
    if (int rc = require_ready()) return rc;
    if (!out) return fail(-1, "NULL output");
    Fields f;
    if (int rc = fields(q, f, from_cons ? "q_cons_vf" : "q_prim_vf")) return rc;
    const Box x = box();
    const Eos e = eos();
    double *dxs[3] = {G.dir[0].ds_dev, G.dir[1].ds_dev, G.dir[2].ds_dev};
    const int nb = cfl_blocks((G.nint + kCflChunk - 1) / kCflChunk);
    if (!partials || nb > capacity)
        return fail(-1, "CFL reduction needs %d partials, the buffer holds %d", nb, capacity);
    const hipStream_t st = G.stream;
    *(volatile uint64_t *)g_result = kPending;
    int rc;
    {
    TimedScope ts(timed ? kKIcfl : -1);
    rc = dispatch_nf_d([&](auto NF, auto D) -> int {
        if (from_cons)
            hipLaunchKernelGGL((k_icfl<decltype(NF)::value, decltype(D)::value, true>), dim3(nb), dim3(kCflThreads), 0,
                               st, f, e, x, dxs[0], dxs[1], dxs[2], dt, G.nint, partials, G.count, g_result);
        else
            hipLaunchKernelGGL((k_icfl<decltype(NF)::value, decltype(D)::value, false>), dim3(nb), dim3(kCflThreads), 0,
                               st, f, e, x, dxs[0], dxs[1], dxs[2], dt, G.nint, partials, G.count, g_result);
        HIPCHK(hipGetLastError());
        return 0;
    });
    }
    if (rc) return rc;
    // The kernel's one store to it, seen as it arrives: the stream's
    // synchronisation returned 5 us later (the call on 200^2 cells 23.6 ->
    // 18.2 us).  The kernels before it on the stream have then ended.  After
    // kPolls looks, a millisecond or two, the call waits for the stream, which
    // also reports errors.
    volatile uint64_t *r = (volatile uint64_t *)g_result;
    for (long n = 0; n < kPolls && *r == kPending; ++n) __builtin_ia32_pause();
    if (*r == kPending) HIPCHK(hipStreamSynchronize(st));
    *out = *(volatile double *)g_result;
    return 0;
}

int mfc_icfl_max(double *const *q_prim_vf, double dt, double *icfl_max) {
    std::lock_guard<std::mutex> reduce(g_reduce);
    return icfl_reduce(q_prim_vf, false, dt, icfl_max, G.partials, kReduceBlocks, true);
}

int mfc_stability_criteria(double *const *q_prim_vf, double dt, double *out) {
    if (!out) return fail(-1, "NULL output");
    out[1] = 0.0;
    out[2] = 0.0;
    std::lock_guard<std::mutex> reduce(g_reduce);
    if (int rc = icfl_reduce(q_prim_vf, false, dt, &out[0], G.partials, kReduceBlocks, true)) return rc;
    if (!G.visc) return 0;
    Fields f;
    if (int rc = fields(q_prim_vf, f, "q_prim_vf")) return rc;
    const Box x = box();
    const Eos e = eos();
    const int nb = (int)std::min<long>(kReduceBlocks, std::max<long>(1, (G.nint + 255) / 256));
    const double *dy = G.D > 1 ? G.dir[1].ds_dev : nullptr;
    int rc = 0;
    if (G.D == 1 || G.D == 2) {
        rc = dispatch_nf_d([&](auto NF, auto D) -> int {
            if constexpr (decltype(D)::value <= 2 && decltype(NF)::value <= kViscFluidsMax) {
                hipLaunchKernelGGL((k_visc_criteria<decltype(NF)::value, decltype(D)::value>), dim3(nb), dim3(256),
                                   0, G.stream, f, e, G.vp, x, G.dir[0].ds_dev, dy, dt, G.nint, G.partials);
                HIPCHK(hipGetLastError());
                return 0;
            } else {
                return fail(-1, "viscous criteria are 1D and 2D only");
            }
        });
    }
    if (rc) return rc;
    double h[2];
    for (int k = 0; k < 2; ++k) {
        hipLaunchKernelGGL(k_reduce_max, dim3(1), dim3(1024), 0, G.stream, G.partials + (long)k * nb, nb);
        HIPCHK(hipGetLastError());
        HIPCHK(hipMemcpyAsync(&h[k], G.partials + (long)k * nb, sizeof(double), hipMemcpyDeviceToHost, G.stream));
    }
    HIPCHK(hipStreamSynchronize(G.stream));
    out[1] = h[0];
    out[2] = -h[1];
    return 0;
}

static int cfl_dt(double *const *q_cons_vf, double cfl, double *dt_out, double *partials, bool timed) {
    if (!(cfl > 0.0)) return fail(-1, "cfl must be positive");
    if (!dt_out) return fail(-1, "NULL output");
    double mx = 0.0;
    std::lock_guard<std::mutex> reduce(g_reduce);
    if (int rc = icfl_reduce(q_cons_vf, true, 1.0, &mx, partials, kReduceBlocks, timed)) return rc;
    if (!(mx > 0.0) || mx != mx) return fail(-5, "CFL reduction gave %g (NaN or non-positive wave speed)", mx);
    *dt_out = cfl / mx;
    return 0;
}

int mfc_cfl_dt(double *const *q_cons_vf, double cfl, double *dt_out) {
    return cfl_dt(q_cons_vf, cfl, dt_out, G.partials, true);
}

int mfc_cfl_dt_noalloc(double *const *q_cons_vf, double cfl, double *dt_out) {
    if (!G.init) return fail(-4, "mfc_rhs_init has not been called");
    return cfl_dt(q_cons_vf, cfl, dt_out, G.scratch, false);
}

int mfc_sizes(int *sys_size, int *buff_size, long *ghost_len, long *interior_len) {
    if (!G.init) return fail(-4, "mfc_rhs_init has not been called");
    if (sys_size) *sys_size = G.S;
    if (buff_size) *buff_size = G.b;
    if (ghost_len) *ghost_len = G.ng;
    if (interior_len) *interior_len = G.nint;
    return 0;
}

int mfc_weno_coefficients(int dir, double *out) {
    if (!G.init) return fail(-4, "mfc_rhs_init has not been called");
    if (dir < 0 || dir >= G.D || !G.dir[dir].ready) return fail(-1, "no grid for direction %d", dir);
    memcpy(out, G.dir[dir].coef_h.data(), sizeof(double) * G.dir[dir].coef_h.size());
    return 0;
}

int mfc_device_alloc(size_t bytes, void **ptr) {
    if (!ptr) return fail(-1, "NULL pointer");
    HIPCHK(hipMalloc(ptr, bytes));
    return 0;
}

int mfc_device_free(void *ptr) {
    HIPCHK(hipFree(ptr));
    return 0;
}

int mfc_memcpy_h2d(void *dst, const void *src, size_t bytes) {
    hipStream_t st = G.init ? G.stream : nullptr;
    HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st));
    HIPCHK(hipStreamSynchronize(st));
    return 0;
}

int mfc_memcpy_d2h(void *dst, const void *src, size_t bytes) {
    hipStream_t st = G.init ? G.stream : nullptr;
    HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    return 0;
}

int mfc_sync(void) {
    if (!G.init) return 0;
    HIPCHK(hipStreamSynchronize(G.stream));
    return 0;
}

void *mfc_stream(void) { return G.init ? (void *)G.stream : nullptr; }

int mfc_timing_enable(int on) {
    if (!G.init) return fail(-4, "mfc_rhs_init has not been called");
    if (int rc = timing_flush()) return rc;
    T.on = on != 0;
    return 0;
}

int mfc_timing_reset(void) {
    if (G.init)
        if (int rc = timing_flush()) return rc;
    for (int k = 0; k < kKCount; ++k) {
        T.total_ms[k] = 0.0;
        T.count[k] = 0;
    }
    return 0;
}

int mfc_timing_read(int kernel, const char **name, double *total_ms, long *count) {
    if (kernel < 0 || kernel >= kKCount) return fail(-1, "kernel id %d outside 0..%d", kernel, kKCount - 1);
    if (G.init)
        if (int rc = timing_flush()) return rc;
    if (name) *name = kKernelNames[kernel];
    if (total_ms) *total_ms = T.total_ms[kernel];
    if (count) *count = T.count[kernel];
    return 0;
}

int mfc_set_stream(void *stream) {
    if (!G.init) return fail(-4, "mfc_rhs_init has not been called");
    G.stream = stream ? (hipStream_t)stream : G.own;
    return 0;
}

int mfc_rhs_finalize(void) {
    if (!G.init) return 0;
    // best-effort teardown: errors here leave nothing to recover
    (void)hipStreamSynchronize(G.stream);
    timing_flush();
    for (auto e : T.pool) (void)hipEventDestroy(e);
    T = Timing();
    for (int d = 0; d < 3; ++d) {
        if (G.dir[d].coef) (void)hipFree(G.dir[d].coef);
        if (G.dir[d].inv_ds) (void)hipFree(G.dir[d].inv_ds);
        if (G.dir[d].ds_dev) (void)hipFree(G.dir[d].ds_dev);
        if (G.dir[d].cc_dev) (void)hipFree(G.dir[d].cc_dev);
        if (G.dir[d].inv_dsg) (void)hipFree(G.dir[d].inv_dsg);
        G.dir[d] = Dir();
    }
    if (G.partials) (void)hipFree(G.partials);
    if (G.scratch_state) (void)hipFree(G.scratch_state);
    if (G.visc_grad) (void)hipFree(G.visc_grad);
    if (G.own) (void)hipStreamDestroy(G.own);
    G = State();
    return 0;
}

} // extern "C"
